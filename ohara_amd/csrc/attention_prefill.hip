// Causal attention over the KV cache for many query positions per sequence (prefill), on MFMA.
//
// Query s of sequence b sits at cache position pos + s and sees positions [0, pos + s]
// (ohara/models/llama.py:100-135: the cache mask key_pos <= start_pos + q_idx :109-113, GQA head
// mapping of repeat_interleave :101-103 by indexing, scale 1/sqrt(Dh), softmax in fp32).
//
// A tile of 64 positions' keys and values travels straight into LDS (global_load_lds), tiles ahead, rows as they lie in the
// cache with their 16-byte pieces permuted by the row's number; for 16 queries of one (sequence, head):
//   S^T = K Q^T   v_mfma_f32_16x16x32_bf16, A = K rows from LDS, B = Q rows held in registers for the whole walk; a lane
//                 ends up with 16 scores of ONE query (its column), so the row max/sum need two cross-lane
//                 steps only;
//   O^T += V^T P  the probabilities go from the scores straight into the B operand (the k-slot -> position
//                 mapping is chosen so that no lane exchange is needed); the A operand - four positions of one
//                 column - is what ds_read_b64_tr_b16 makes of four rows of V: within sixteen lanes, lane 4 r + c
//                 reads columns 4 c .. 4 c + 3 of row r and lane n receives column n of the four rows.
// The running max / sum / rescale are the usual online softmax; probabilities are rounded to bf16 for the second product,
// sums are kept in fp32, positions are added in their order whatever the shape of the workgroup.
//
// Four kernels: one wave per 16 or 32 queries where there are many (attn_flow_kernel, attn_prefill_kernel), four waves per 16 where there are
// few and the walk over the positions is a chain (attn_team_kernel), and for few queries behind a long context - with room for partial
// results from the caller - the positions in chunks, each a workgroup's (attn_chunk_kernel).
//
// What bounds them: the softmax between the products, and where the keys and values come from.  A head's q blocks read
// the same ones: spread round-robin over the XCDs every L2 held every head's, and the launch waited for memory.
#include "lds_tile.h"

#include <algorithm>

namespace {

struct PrefillArgs {
  const bf16_t* q;   // (B*S, H*D)
  const bf16_t* k;   // (Bcap, Tmax, Hkv, D)
  const bf16_t* v;
  bf16_t* out;       // (B*S, H*D)
  int B, S, H, Hkv, Tmax, pos;
  int nqb;           // query blocks per sequence
  float scale_log2e;
  const int32_t* seqs;  // prompts of their own lengths, from position 0: B first rows, B lengths, B rows of the cache (S: the longest)
};
struct Sequence {
  size_t row0;  // first query row
  int S, cache;
};
__device__ __forceinline__ Sequence sequence(const PrefillArgs& a, int b) {
  if (a.seqs) return {(size_t)a.seqs[b], a.seqs[a.B + b], a.seqs[2 * a.B + b]};
  return {(size_t)b * a.S, a.S, b};
}

// An XCD (ids go round-robin over the eight) gets whole heads, their late - longest - blocks first; where the heads do
// not divide, an eighth of all blocks in the order of the heads, long and short ones in turn.  Where the sequences have lengths of
// their own every eighth head, so that no XCD gets the long ones; the grid is rounded up to that (then head may be past the last).
__device__ __forceinline__ void my_block(const PrefillArgs& a, int& head, int& qblk) {
  const int heads = a.H * a.B, x = blockIdx.x & 7, q = blockIdx.x >> 3;
  if (a.seqs) {
    const int nh = (heads + 7) >> 3;
    head = (q % nh) * 8 + x;
    qblk = a.nqb - 1 - q / nh;
  } else if ((heads & 7) == 0) {
    const int nh = heads >> 3;
    head = x * nh + q % nh;
    qblk = a.nqb - 1 - q / nh;
  } else {
    const int n = gridDim.x, p = x * (n >> 3) + min(x, n & 7) + q;
    head = p / a.nqb;
    const int r = p - head * a.nqb;
    qblk = r & 1 ? r >> 1 : a.nqb - 1 - (r >> 1);
  }
}

constexpr int KT = 64;                // positions of a tile
constexpr int NKB = KT / 16, NWIN = KT / 32;

// A tile in LDS: the keys' rows, then the values'.  How NW waves bring it there, and where a lane finds its fragments.
template <int D>
struct KvTile {
  static constexpr int ROWB = 2 * D, PIECES = ROWB / 16, RPL = 1024 / ROWB;  // bytes and 16-byte pieces of a row, rows of a load
  static constexpr int BYTES = KT * ROWB, SLOT = 2 * BYTES;
  const char *kb, *vb;  // the sequence's first row of this head
  uint32_t rowb;        // bytes from one position to the next
  int len;              // positions that exist
  int lane;

  __device__ __forceinline__ KvTile(const PrefillArgs& a, const Sequence& sq, int kvh, int lane_) : lane(lane_) {
    const size_t row = (size_t)a.Hkv * D;
    kb = reinterpret_cast<const char*>(a.k + (size_t)sq.cache * a.Tmax * row + (size_t)kvh * D);
    vb = reinterpret_cast<const char*>(a.v + (size_t)sq.cache * a.Tmax * row + (size_t)kvh * D);
    rowb = (uint32_t)row * 2;
    len = a.pos + sq.S;
  }
  // ALIGNED: the caches start on 16 bytes (false: through registers, any)
  template <int NW>
  struct Offsets {
    static_assert(KT / RPL % NW == 0, "loads split evenly over the waves");
    static constexpr int N = KT / RPL / NW;
    uint32_t k[N], v[N];
  };
  // this lane's of the loads of a tile that holds `rows` positions: past them, the last one (masked)
  template <int NW>
  __device__ __forceinline__ Offsets<NW> offsets(int rows, int wave) const {
    Offsets<NW> o;
    const int lr = lane / PIECES, lq = lane % PIECES;  // its row of a load, and its place in it
#pragma unroll
    for (int i = 0; i < o.N; ++i) {
      const int r = (wave + i * NW) * RPL + lr;
      const uint32_t ro = (uint32_t)min(r, rows - 1) * rowb;
      o.k[i] = ro + (uint32_t)((lq ^ r) & (PIECES - 1)) * 16;
      o.v[i] = ro + (uint32_t)(lq ^ ((r & (PIECES / 2 - 1)) << 1)) * 16;
    }
    return o;
  }
  template <int NW, bool ALIGNED>
  __device__ __forceinline__ void issue(int t, uint32_t slot, int wave, const Offsets<NW>& full) const {
    const char* kt = kb + (size_t)(t * KT) * rowb;
    const char* vt = vb + (size_t)(t * KT) * rowb;
    Offsets<NW> o = full;
    if (t * KT + KT > len) o = offsets<NW>(len - t * KT, wave);
#pragma unroll
    for (int i = 0; i < o.N; ++i) {
      const uint32_t dst = slot + (wave + i * NW) * 1024;
      if (ALIGNED) {
        load_lds16(dst, kt, o.k[i]);
        load_lds16(dst + BYTES, vt, o.v[i]);
      } else {
        const uint4 kv = ldg16(kt + o.k[i]), vv = ldg16(vt + o.v[i]);
        *(OHARA_LDS u32x4*)(uintptr_t)(dst + lane * 16) = (u32x4){kv.x, kv.y, kv.z, kv.w};
        *(OHARA_LDS u32x4*)(uintptr_t)(dst + BYTES + lane * 16) = (u32x4){vv.x, vv.y, vv.z, vv.w};
      }
    }
  }
  // one half of a tile, its keys or its values, whose first load of a full tile is at `off`
  template <int NW, bool KEYS>
  __device__ __forceinline__ void issue_half(int t, uint32_t at, int wave, uint32_t off) const {
    constexpr int N = KT / RPL / NW, STEP = NW * RPL;  // a wave's loads, positions between them: whole periods of the permutation
    static_assert(STEP % PIECES == 0, "");
    const char* from = (KEYS ? kb : vb) + (size_t)(t * KT) * rowb;
    if (t * KT + KT <= len) {
#pragma unroll
      for (int i = 0; i < N; ++i) load_lds16(at + (wave + i * NW) * 1024, from + (size_t)(i * STEP) * rowb, off);
    } else {
      int rows = len - t * KT;
      asm volatile("" : "+s"(rows));  // (else every tile works these out, for the last one)
      const Offsets<NW> o = offsets<NW>(rows, wave);
#pragma unroll
      for (int i = 0; i < N; ++i) load_lds16(at + (wave + i * NW) * 1024, from, KEYS ? o.k[i] : o.v[i]);
    }
  }
  // keys of positions 16 kb + (lane & 15), columns 32 j + 8 (lane >> 4) .. + 7
  __device__ __forceinline__ uint4 keys(uint32_t slot, int kb_, int j) const {
    const int m = lane & 15, g = lane >> 4;
    return lds16_at(slot + (16 * kb_ + m) * ROWB + (uint32_t)((4 * j + g) ^ (m & (PIECES - 1))) * 16);
  }
  // column 16 d + (lane & 15) of the values of positions 32 w + 4 g .. + 3 and of those 16 later
  __device__ __forceinline__ uint4 values(uint32_t slot, int w, int d) const {
    const int m = lane & 15, row = 4 * (lane >> 4) + (m >> 2);
    const uint32_t at = slot + BYTES + (32 * w + row) * ROWB + (m & 3) * 8 + (uint32_t)((row & (PIECES / 2 - 1)) ^ d) * 32;
    const uint2 lo = lds_tr8(at), hi = lds_tr8(at + 16 * ROWB);
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
  }
};

template <bool ALIGNED, int LEFT>
__device__ __forceinline__ void tile_barrier() {  // this wave's older loads have landed, and everyone's
  if (ALIGNED) wait_loads<LEFT>();
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
}

// Online softmax over a tile, per query (= per lane column).  The running maximum is kept as an integer (log2 units): every rescale
// is then an exact power of two and the bf16 weights do not depend on which tile raised it (common.h: softmax bookkeeping).
struct Shift {
  float off, corr;  // a weight's exponent is score * mul - off; what the sums so far are multiplied with
};
__device__ __forceinline__ Shift softmax_shift(float tmax, float& m_run) {  // tmax: this lane's
  tmax = lane_xor_max<32>(lane_xor_max<16>(tmax));
  const float mn = fmaxf(m_run, ceilf(tmax));
  const float corr = pow2_neg_int(m_run - mn);
  m_run = mn;
  return {mn == -INFINITY ? 0.f : mn, corr};  // (a chunk may begin behind the last position of a query: all its weights are zeros)
}
__device__ __forceinline__ void softmax_mask(f32x4 (&s)[NKB], int t0, int qpos, int g, float scale_log2e) {
#pragma unroll
  for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = s[kk][i] * scale_log2e;
      s[kk][i] = t0 + kk * 16 + 4 * g + i > qpos ? -INFINITY : v;
    }
}
__device__ __forceinline__ void softmax_weights(const f32x4 (&s)[NKB], float mul, const Shift& x, uint4 (&pf)[NWIN], float& l_run) {
  float ts = 0.f;
  float p[NKB][4];
#pragma unroll
  for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[kk][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kk][i], mul, -x.off));
      ts += p[kk][i];
    }
  l_run = l_run * x.corr + ts;  // this lane's share; lanes g = 0..3 are added at the end
  // k-slot 8 g + i of window w  <->  position 32 w + 4 g + i (i < 4), 32 w + 16 + 4 g + i - 4
#pragma unroll
  for (int w = 0; w < NWIN; ++w)
    pf[w] = make_uint4(pack_bf(p[2 * w][0], p[2 * w][1]), pack_bf(p[2 * w][2], p[2 * w][3]),
                       pack_bf(p[2 * w + 1][0], p[2 * w + 1][1]), pack_bf(p[2 * w + 1][2], p[2 * w + 1][3]));
}
// s -> the B operand of the second product; the result multiplies the accumulators
__device__ __forceinline__ float softmax_tile(f32x4 (&s)[NKB], uint4 (&pf)[NWIN], float& m_run, float& l_run, int t0, int first, int qpos,
                                              int g, float scale_log2e) {
  float mul = scale_log2e;        // what the stored scores still have to be multiplied with: in the exponent's fused multiply-add
  if (t0 + KT - 1 > first) {      // (wave-uniform) the tile reaches past the wave's first query
    softmax_mask(s, t0, qpos, g, scale_log2e);
    mul = 1.0f;
  }
  float tmax = -INFINITY;
#pragma unroll
  for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
    for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[kk][i]);
  const Shift x = softmax_shift(tmax * mul, m_run);  // the scale is positive: the maximum of the products is the product of the maximum
  softmax_weights(s, mul, x, pf, l_run);
  return x.corr;
}

// Queries wq0 + 16 qb + (lane & 15): lane g holds columns 32 j + 8 g .. + 7
template <int D>
__device__ __forceinline__ void load_queries(uint4 (&qf)[D / 32], int& qpos, const PrefillArgs& a, const Sequence& sq, int h, int qi, int g) {
  qpos = qi < sq.S ? a.pos + qi : 0x3fffffff;  // rows past the end: never masked, never stored
#pragma unroll
  for (int j = 0; j < D / 32; ++j)
    qf[j] = qi < sq.S ? ldg16(a.q + (sq.row0 + qi) * a.H * D + (size_t)h * D + 32 * j + 8 * g) : make_uint4(0, 0, 0, 0);
}

template <int D, int N>
__device__ __forceinline__ void store_rows(const f32x4 (&o)[N], float l, const PrefillArgs& a, const Sequence& sq, int h, int qi, int g, int d0) {
  l = lane_xor_sum<32>(lane_xor_sum<16>(l));
  if (qi >= sq.S) return;
  const float inv = 1.0f / l;
  bf16_t* dst = a.out + (sq.row0 + qi) * a.H * D + (size_t)h * D + 16 * d0 + 4 * g;
#pragma unroll
  for (int db = 0; db < N; ++db)
    *reinterpret_cast<uint2*>(dst + db * 16) = make_uint2(pack_bf(o[db][0] * inv, o[db][1] * inv), pack_bf(o[db][2] * inv, o[db][3] * inv));
}

// Two to fifteen tokens a call (FEW).  A masked position weighs zero in a tile, and zero times an infinity is a NaN, for queries that do not
// see it: calls of more tokens live with that (so does softmax(...) @ v); these went through kernels that walk each token's own positions
// and still give such kernels' results.  So a query whose sums are not finite walks its positions once more, by itself: the weights are
// the same bits times a power of two (common.h: softmax bookkeeping).  That costs nothing where sums are finite; taking the masked values out of
// the products, where a product with zeros says that it is needed, cost every call 0.3 to 0.6 us, or a tenth (8 x 15 behind 3000).
// The queries q0 + m with a bit in `which` -> columns c0 .. c0 + cols - 1 of their rows.
template <int D>
__device__ __forceinline__ void walk_rows(const PrefillArgs& a, const Sequence& sq, int h, int q0, unsigned int which, int c0, int cols, int lane) {
  constexpr int N = D / 64, AT = 8;  // columns of a lane, positions at a time
  const size_t row = (size_t)a.Hkv * D, at0 = (size_t)sq.cache * a.Tmax * row + (size_t)(h / (a.H / a.Hkv)) * D + lane;
#pragma unroll 1
  for (int m = 0; m < 16 && q0 + m < sq.S; ++m) {
    if (!(which >> m & 1)) continue;
    const size_t mine = (sq.row0 + q0 + m) * a.H * D + (size_t)h * D + lane;
    const int last = a.pos + q0 + m;
    float x[N], o[N], top = -INFINITY, l = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      x[i] = bf2f(a.q[mine + 64 * i]);
      o[i] = 0.f;
    }
#pragma unroll 1
    for (int p0 = 0; p0 <= last; p0 += AT) {
      bf16_t k[AT][N], v[AT][N];
#pragma unroll
      for (int j = 0; j < AT; ++j)
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const size_t at = at0 + (size_t)min(p0 + j, last) * row + 64 * i;
          k[j][i] = a.k[at];
          v[j][i] = a.v[at];
        }
#pragma unroll
      for (int j = 0; j < AT; ++j) {
        if (p0 + j > last) break;
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < N; ++i) s = __builtin_fmaf(x[i], bf2f(k[j][i]), s);
        s = wave_sum(s) * a.scale_log2e;
        const float higher = fmaxf(top, ceilf(s)), back = pow2_neg_int(top - higher);
        top = higher;
        const float w = __builtin_amdgcn_exp2f(s - (top == -INFINITY ? 0.f : top));
        l = l * back + w;
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = o[i] * back + rbf(w) * bf2f(v[j][i]);
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (lane + 64 * i >= c0 && lane + 64 * i < c0 + cols) a.out[mine + 64 * i] = f2bf(o[i] * (1.0f / l));
  }
}
// ... and the rest as they are.
template <int D, int N>
__device__ __forceinline__ void store_few(const f32x4 (&o)[N], float l, const PrefillArgs& a, const Sequence& sq, int h, int q0, int lane, int d0) {
  float sum = 0.f;
#pragma unroll
  for (int db = 0; db < N; ++db) sum += (o[db][0] + o[db][1]) + (o[db][2] + o[db][3]);
  const unsigned int odd = columns_not_finite(sum);
  store_rows<D>(o, l, a, sq, h, odd >> (lane & 15) & 1 ? sq.S : q0 + (lane & 15), lane >> 4, d0);
  if (odd) walk_rows<D>(a, sq, h, q0, odd, 16 * d0, 16 * N, lane);
}

// Four waves of 16 QW queries, one tile ahead, scores, softmax and values one after the other.  With heads of 128 a wave that adds values goes
// before the other of its SIMD, which keeps the two apart: 32 queries a wave, us without / with: 4001 x 32 heads (8 KV heads) 189 / 180, 4 x 2048
// x 16 (4) 100.5 / 93, 16 x 700 x 16 (4) 74.1 / 71.6 (heads of 64: no difference).
template <int D, int QW, bool ALIGNED, bool FEW>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(PrefillArgs a) {
  constexpr int NW = 4, QB = 16 * QW * NW;
  static_assert(!FEW || QW == 1, "sixteen queries a wave");
  constexpr int NK = D / 32;             // k-steps of the score product
  constexpr int ND = D / 16;             // 16-column blocks of the output
  typedef KvTile<D> Tl;
  extern __shared__ __align__(16) unsigned char smem[];
  int head, qblk;
  my_block(a, head, qblk);
  const int b = head / a.H, h = head - b * a.H;
  if (b >= a.B) return;
  const Sequence sq = sequence(a, b);
  if (qblk * QB >= sq.S) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int q0 = qblk * QB;                              // first query of the workgroup
  const int wq0 = q0 + wave * 16 * QW;                   // first query of the wave
  const Tl tile(a, sq, h / (a.H / a.Hkv), lane);
  const typename Tl::template Offsets<NW> offs = tile.template offsets<NW>(KT, wave);
  const int ntiles = (min(a.pos + q0 + QB, tile.len) + KT - 1) / KT;  // tiles any query of the workgroup sees
  const int wave_last = min(a.pos + wq0 + 16 * QW - 1, tile.len - 1);  // last position any query of the wave sees
  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;

  uint4 qf[QW][NK];
  int qpos[QW];
  f32x4 o[QW][ND];
  float m_run[QW], l_run[QW];
#pragma unroll
  for (int qb = 0; qb < QW; ++qb) {
    load_queries<D>(qf[qb], qpos[qb], a, sq, h, wq0 + qb * 16 + m, g);
    m_run[qb] = -INFINITY;
    l_run[qb] = 0.f;
#pragma unroll
    for (int db = 0; db < ND; ++db) o[qb][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  tile.template issue<NW, ALIGNED>(0, lds0, wave, offs);
  uint32_t cur = lds0;
  for (int t = 0; t < ntiles; ++t) {
    tile_barrier<ALIGNED, 0>();  // the tile is there, and everyone is done with the one before
    const uint32_t next = lds0 + Tl::SLOT - (cur - lds0);
    if (t + 1 < ntiles) tile.template issue<NW, ALIGNED>(t + 1, next, wave, offs);
    const int t0 = t * KT;
    if (t0 <= wave_last) {  // else wholly masked for this wave (barriers stay uniform)
      // all fragments read before the first product, and the products of different blocks in turn, so that none waits
      // for the one before it
      f32x4 s[QW][NKB];
      uint4 kf[NKB][NK];
#pragma unroll
      for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
        for (int j = 0; j < NK; ++j) kf[kk][j] = tile.keys(cur, kk, j);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NK; ++j)
#pragma unroll
        for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
          for (int qb = 0; qb < QW; ++qb)
            s[qb][kk] = mfma16(kf[kk][j], qf[qb][j], j ? s[qb][kk] : (f32x4){0.f, 0.f, 0.f, 0.f});
      __builtin_amdgcn_sched_barrier(0);
      uint4 pf[QW][NWIN];
#pragma unroll
      for (int qb = 0; qb < QW; ++qb) {
        const float corr = softmax_tile(s[qb], pf[qb], m_run[qb], l_run[qb], t0, a.pos + wq0 + 16 * qb, qpos[qb], g, a.scale_log2e);
        if (__any(corr != 1.0f)) {  // most tiles leave the running maximum of every query of the wave alone
#pragma unroll
          for (int db = 0; db < ND; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[qb][db][i] *= corr;
        }
      }
      if (D == 128) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int w = 0; w < NWIN; ++w) {
        uint4 vf[ND];  // all read before the first product, as above
#pragma unroll
        for (int db = 0; db < ND; ++db) vf[db] = tile.values(cur, w, db);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int db = 0; db < ND; ++db)
#pragma unroll
          for (int qb = 0; qb < QW; ++qb) o[qb][db] = mfma16(vf[db], pf[qb][w], o[qb][db]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (D == 128) __builtin_amdgcn_s_setprio(0);
    }
    cur = next;
  }
  if constexpr (FEW) return store_few<D>(o[0], l_run[0], a, sq, h, wq0, lane, 0);
#pragma unroll
  for (int qb = 0; qb < QW; ++qb) store_rows<D>(o[qb], l_run[qb], a, sq, h, wq0 + qb * 16 + m, g, 0);
}

// Four waves of 16 queries.  While tile t + 1 is scored the weights of tile t are made, and while the values of t are added the maxima of t + 1
// are found: in one wave the products and the softmax keep both units busy, where one after the other (the kernel above) they leave each
// idle in turn and only another wave fills in.  All of a round's fragments are read before its first product; in the second half, which
// is mostly products, a wave goes before the other of its SIMD, so that the two fall into different halves (4001 x 16 heads, 4 KV
// heads, of 128: 93.2 us without, 91.5 with).  us, one after the other / this: 1024 x 16 25.8 / 21.9, 2048 x 6 45.7 / 36.0, 2048 x 16
// 48.6 / 40.3, 3001 x 16 71.7 / 58.4, 4001 x 16 103.9 / 91.5, 32 x 300 x 6 behind 1500 115 / 92; heads of 64, 4001 x 16 68.8 / 55.7.
// 238 VGPRs: 32 queries a wave do not fit (with fragments in parts of two they spill ten: 2048 x 6 55.6).
template <int D, bool CHUNK>  // CHUNK: tiles first .. end - 1 of a walk; else from the start to the last that any query sees
__device__ __forceinline__ void flow_walk(const KvTile<D>& tile, int first, int end, int wave, const uint4 (&qf)[D / 32], int qpos,
                                          int q_first /* the wave's first query's position */, int wave_last, uint32_t lds0, float scale_log2e,
                                          f32x4 (&o)[D / 16], float& m_run, float& l_run) {
  constexpr int NW = 4, NK = D / 32, ND = D / 16;
  typedef KvTile<D> Tl;
  constexpr int BY = Tl::BYTES, LOADS = KT / Tl::RPL / NW;
  const int m = tile.lane & 15, g = tile.lane >> 4;
  const typename Tl::template Offsets<NW> offs = tile.template offsets<NW>(KT, wave);
  const uint32_t koff = offs.k[0], voff = offs.v[0];
#pragma unroll
  for (int db = 0; db < ND; ++db) o[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  m_run = -INFINITY;
  l_run = 0.f;
  if (CHUNK && first >= end) return;
  tile.template issue_half<NW, true>(first, lds0, wave, koff);
  tile.template issue_half<NW, false>(first, lds0 + 2 * BY, wave, voff);
  if (first + 1 < end) tile.template issue_half<NW, true>(first + 1, lds0 + BY, wave, koff);

  // where this lane's fragments lie (KvTile::keys and ::values): the permutations are an exclusive or
  const uint32_t kp = m * Tl::ROWB + (uint32_t)(g ^ (m & (Tl::PIECES - 1))) * 16;
  const int vr = 4 * g + (m >> 2);
  const uint32_t vp = vr * Tl::ROWB + (m & 3) * 8 + (uint32_t)(vr & (Tl::PIECES / 2 - 1)) * 32;
  auto read_keys = [&](uint4 (&kf)[NK][NKB], uint32_t at) {
#pragma unroll
    for (int j = 0; j < NK; ++j)
#pragma unroll
      for (int kk = 0; kk < NKB; ++kk) kf[j][kk] = lds16_at((kp ^ (j * 64)) + (at + kk * (16 * Tl::ROWB)));
  };
  auto read_values = [&](uint4 (&vf)[NWIN][ND], uint32_t at) {
#pragma unroll
    for (int w = 0; w < NWIN; ++w)
#pragma unroll
      for (int db = 0; db < ND; ++db) {
        const uint32_t p = vp ^ (db * 32), from = at + w * (32 * Tl::ROWB);
        const uint2 lo = lds_tr8(p + from), hi = lds_tr8(p + (from + 16 * Tl::ROWB));
        vf[w][db] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
  };
  auto score = [&](f32x4 (&r)[NKB], const uint4 (&kf)[NK][NKB]) {
#pragma unroll
    for (int j = 0; j < NK; ++j)
#pragma unroll
      for (int kk = 0; kk < NKB; ++kk) r[kk] = mfma16(kf[j][kk], qf[j], j ? r[kk] : (f32x4){0.f, 0.f, 0.f, 0.f});
  };
  f32x4 s[NKB];  // tile t's scores, what they have to be multiplied with, and their maximum's shift
  float mul;
  Shift x;
  if (CHUNK) {
    mul = 1.0f;
    x = {0.f, 1.f};
  }
  auto shift = [&] {
    float top = -INFINITY;
#pragma unroll
    for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i) top = fmaxf(top, s[kk][i]);
    x = softmax_shift(top * mul, m_run);
  };
  auto add = [&](const uint4 (&vf)[NWIN][ND], const uint4 (&pf)[NWIN]) {
#pragma unroll
    for (int w = 0; w < NWIN; ++w)
#pragma unroll
      for (int db = 0; db < ND; ++db) o[db] = mfma16(vf[w][db], pf[w], o[db]);
  };

  if (first + 1 < end) tile_barrier<true, 2 * LOADS>();
  else tile_barrier<true, LOADS>();
  if (!CHUNK || first * KT <= wave_last) {
    uint4 kf[NK][NKB];
    read_keys(kf, lds0);
    score(s, kf);
    const bool masked = first * KT + KT - 1 > q_first;
    if (masked) softmax_mask(s, first * KT, qpos, g, scale_log2e);
    mul = masked ? 1.0f : scale_log2e;
    shift();
  }
  auto round = [&](int t, auto parity) {
    constexpr int P = decltype(parity)::value;
    tile_barrier<true, 0>();  // the next keys and these values are there, and everyone is done with those before
    if (t + 2 < end) tile.template issue_half<NW, true>(t + 2, lds0 + P * BY, wave, koff);
    if (t + 1 < end) tile.template issue_half<NW, false>(t + 1, lds0 + (3 - P) * BY, wave, voff);
    const int t1 = (t + 1) * KT;
    uint4 vf[NWIN][ND], pf[NWIN];
    auto flow = [&](auto masked) {  // masked: not every query of the wave sees the whole of tile t + 1
      uint4 kf[NK][NKB];
      f32x4 sn[NKB];
      read_keys(kf, lds0 + (1 - P) * BY);
      read_values(vf, lds0 + (2 + P) * BY);
      __builtin_amdgcn_sched_barrier(0);
      score(sn, kf);
      softmax_weights(s, mul, x, pf, l_run);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < NKB; ++kk) s[kk] = sn[kk];
      mul = decltype(masked)::value ? 1.0f : scale_log2e;
      if (decltype(masked)::value) softmax_mask(s, t1, qpos, g, scale_log2e);
      __builtin_amdgcn_s_setprio(1);
      __builtin_amdgcn_sched_barrier(0);
      add(vf, pf);
      shift();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
      if (__any(x.corr != 1.0f)) {  // most tiles leave the running maximum of every query of the wave alone
#pragma unroll
        for (int db = 0; db < ND; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[db][i] *= x.corr;
      }
    };
    const bool more = !CHUNK || t + 1 < end;  // (all of these are wave-uniform)
    if (more && t1 + KT - 1 <= q_first) {
      flow(std::false_type());
    } else if (more && t1 <= wave_last) {
      flow(std::true_type());
    } else if (t * KT <= wave_last) {  // the wave's last tile
      read_values(vf, lds0 + (2 + P) * BY);
      softmax_weights(s, mul, x, pf, l_run);
      add(vf, pf);
    }
  };
  for (int t = first; t < end; t += 2) {
    round(t, std::integral_constant<int, 0>());
    if (t + 1 < end) round(t + 1, std::integral_constant<int, 1>());
  }
}
template <int D>
__global__ __launch_bounds__(256, 2) void attn_flow_kernel(PrefillArgs a) {
  constexpr int NW = 4, QB = 16 * NW, NK = D / 32, ND = D / 16;
  typedef KvTile<D> Tl;
  extern __shared__ __align__(16) unsigned char smem[];
  int head, qblk;
  my_block(a, head, qblk);
  const int b = head / a.H, h = head - b * a.H;
  if (b >= a.B) return;
  const Sequence sq = sequence(a, b);
  if (qblk * QB >= sq.S) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int q0 = qblk * QB, wq0 = q0 + wave * 16;
  const Tl tile(a, sq, h / (a.H / a.Hkv), lane);
  const int ntiles = (min(a.pos + q0 + QB, tile.len) + KT - 1) / KT;   // tiles any query of the workgroup sees
  const int wave_last = min(a.pos + wq0 + 15, tile.len - 1);           // last position any query of the wave sees
  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;  // keys of even and of odd tiles, then their values

  uint4 qf[NK];
  int qpos;
  load_queries<D>(qf, qpos, a, sq, h, wq0 + m, g);
  f32x4 o[ND];
  float m_run, l_run;
  flow_walk<D, false>(tile, 0, ntiles, wave, qf, qpos, a.pos + wq0, wave_last, lds0, a.scale_log2e, o, m_run, l_run);
  store_rows<D>(o, l_run, a, sq, h, wq0 + m, g, 0);
}

// TEAMS teams of four waves, 16 queries each.  Wave w scores positions 16 w .. + 15 of every tile and owns a quarter of the output
// columns; the scores go through LDS, and every wave of the team does the softmax of the whole tile.  In the round that works
// off tile t the scores of t + 1 are made: one barrier a tile.
template <int D, int TEAMS, int NST, bool ALIGNED, bool FEW>
__global__ __launch_bounds__(TEAMS * 256, TEAMS) void attn_team_kernel(PrefillArgs a) {
  constexpr int NW = 4 * TEAMS, QB = 16 * TEAMS;
  constexpr int NK = D / 32, ND = D / 64;  // k-steps of the score product, 16-column blocks of a wave's output
  typedef KvTile<D> Tl;
  constexpr int LPW = 2 * KT / Tl::RPL / NW;  // a wave's loads of a tile
  extern __shared__ __align__(16) unsigned char smem[];
  int head, qblk;
  my_block(a, head, qblk);
  const int b = head / a.H, h = head - b * a.H;
  if (b >= a.B) return;
  const Sequence sq = sequence(a, b);
  if (qblk * QB >= sq.S) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w4 = wave & 3, team = wave >> 2;
  const int m = lane & 15, g = lane >> 4;
  const int q0 = qblk * QB, wq0 = q0 + 16 * team;
  const Tl tile(a, sq, h / (a.H / a.Hkv), lane);
  const typename Tl::template Offsets<NW> offs = tile.template offsets<NW>(KT, wave);
  const int ntiles = (min(a.pos + q0 + QB, tile.len) + KT - 1) / KT;
  const int team_last = min(a.pos + wq0 + 15, tile.len - 1);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;
  const uint32_t sc0 = lds0 + NST * Tl::SLOT + team * 4096 + lane * 16;  // the team's scores: two tiles' in turn

  uint4 qf[NK];
  int qpos;
  load_queries<D>(qf, qpos, a, sq, h, wq0 + m, g);
  f32x4 o[ND];
#pragma unroll
  for (int db = 0; db < ND; ++db) o[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  auto scores = [&](const uint4 (&kf)[NK]) {
    f32x4 s = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NK; ++j) s = mfma16(kf[j], qf[j], s);
    return s;
  };
  auto put_scores = [&](int t, f32x4 s) { *(OHARA_LDS f32x4*)(uintptr_t)(sc0 + (t & 1) * (TEAMS * 4096) + w4 * 1024) = s; };

#pragma unroll
  for (int t = 0; t < NST - 1; ++t)
    if (t < ntiles) tile.template issue<NW, ALIGNED>(t, lds0 + t * Tl::SLOT, wave, offs);
  if (NST - 2 < ntiles) tile_barrier<ALIGNED, (NST - 2) * LPW>();
  else tile_barrier<ALIGNED, 0>();
  uint4 kf[NK];
#pragma unroll
  for (int j = 0; j < NK; ++j) kf[j] = tile.keys(lds0, w4, j);
  put_scores(0, scores(kf));
  uint32_t cur = lds0;
  for (int t = 0; t < ntiles; ++t) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the scores of this tile are written
    if (t + NST - 2 < ntiles) tile_barrier<ALIGNED, (NST - 3) * LPW>();  // and the next tile is there
    else tile_barrier<ALIGNED, 0>();
    asm volatile("" ::: "memory");
    const uint32_t next = cur + Tl::SLOT == lds0 + NST * Tl::SLOT ? lds0 : cur + Tl::SLOT;
    if (t + NST - 1 < ntiles) tile.template issue<NW, ALIGNED>(t + NST - 1, cur == lds0 ? lds0 + (NST - 1) * Tl::SLOT : cur - Tl::SLOT, wave, offs);
    const int t0 = t * KT;
    // everything this round reads, then the products (past the last tile: of what the slot holds, unused)
    f32x4 s[NKB];
    uint4 vf[NWIN][ND];
#pragma unroll
    for (int kk = 0; kk < NKB; ++kk) s[kk] = *(OHARA_LDS f32x4*)(uintptr_t)(sc0 + (t & 1) * (TEAMS * 4096) + kk * 1024);
#pragma unroll
    for (int j = 0; j < NK; ++j) kf[j] = tile.keys(next, w4, j);
#pragma unroll
    for (int w = 0; w < NWIN; ++w)
#pragma unroll
      for (int db = 0; db < ND; ++db) vf[w][db] = tile.values(cur, w, w4 * ND + db);
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 sn = scores(kf);
    if (TEAMS == 1 || t0 <= team_last) {  // else wholly masked for this team
      uint4 pf[NWIN];
      const float corr = softmax_tile(s, pf, m_run, l_run, t0, a.pos + wq0, qpos, g, a.scale_log2e);
#pragma unroll
      for (int db = 0; db < ND; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[db][i] *= corr;
#pragma unroll
      for (int w = 0; w < NWIN; ++w)
#pragma unroll
        for (int db = 0; db < ND; ++db) o[db] = mfma16(vf[w][db], pf[w], o[db]);
    }
    put_scores(t + 1, sn);
    cur = next;
  }
  if constexpr (FEW) return store_few<D>(o, l_run, a, sq, h, wq0, lane, w4 * ND);
  store_rows<D>(o, l_run, a, sq, h, wq0 + m, g, w4 * ND);
}

// Few queries behind a long context.  What bounds the kernels above there is a CU's rate of taking in keys and values, 50 GB/s: 1.5 MB a
// head at 3000 positions are 31 us, however its waves share them.  So a workgroup takes a chunk of the positions, for four tasks of
// one KV head - a task is 16 queries of one head; the heads of a group come first, they see the same positions - a wave each, and leaves
// partial sums for attn_chunks_merge_kernel.  us with both launches, the kernels above / these: 16 queries x 16 heads (4 KV heads) of
// 128 behind 3000 34.5 / 10.8, 48 queries 35.1 / 13.0, 200 38.4 / 22.5; 4 x 48 behind 1900 25.1 / 17.3; 200 x 16 heads of 64 behind
// 2000 21.6 / 13.5.
// The walk over a chunk is attn_flow_kernel's; one after the other / so: 4 x 48 behind 1900 21.4 / 20.5, 4 x 200 behind 2000 42.4 / 39.5, 200 behind 3000
// 27.6 / 25.9, 8 x 100 x 6 heads behind 3000 34.3 / 33.2 (on a slower card than the lines above).  Waves without a task (up to 16 queries of a KV head of
// its own leave three) only load: 8 x 16 x 6 heads behind 3000 27.9 one after the other, 27.2 with them walking too, 26.9; 4 x 16 x 16 32.2, 31.1, 30.6.
struct Cut {
  int tasks, ntb, chunks, tiles;  // tasks of a (sequence, KV head) and fours of them; chunks, and tiles of one
};
struct ChunkArgs {
  PrefillArgs p;
  Cut cut;
  int group;    // heads a KV head
  float* part;  // [task][chunk]: 16 D sums in lane order, 16 maxima, 16 sums of the weights
};

template <int D>
__global__ __launch_bounds__(256, 2) void attn_chunk_kernel(ChunkArgs c) {
  constexpr int NW = 4, NK = D / 32, ND = D / 16, PS = 16 * D + 32;
  typedef KvTile<D> Tl;
  extern __shared__ __align__(16) unsigned char smem[];
  const PrefillArgs& a = c.p;
  // an XCD gets neighbouring workgroups: the chunks and fours of one KV head share its L2
  const int n = c.p.B * c.p.Hkv * c.cut.ntb * c.cut.chunks, xcd = blockIdx.x & 7, share = (n + 7) >> 3;
  const int id = xcd * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || id >= n) return;
  const int tb = id % c.cut.ntb, chunk = id / c.cut.ntb % c.cut.chunks, bh = id / (c.cut.ntb * c.cut.chunks), b = bh / a.Hkv, kvh = bh - b * a.Hkv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int task = tb * NW + wave, last_task = min(tb * NW + NW, c.cut.tasks) - 1;
  const int wq0 = task / c.group * 16, h = kvh * c.group + task % c.group;
  const Sequence sq = sequence(a, b);
  const Tl tile(a, sq, kvh, lane);
  const int first = chunk * c.cut.tiles, seen = (min(a.pos + last_task / c.group * 16 + 16, tile.len) + KT - 1) / KT;
  const int end = min(first + c.cut.tiles, seen);                           // tiles any task of the workgroup sees
  const bool mine = task < c.cut.tasks;  // (a wave without a task only loads: it sees no position)
  const int wave_first = mine ? a.pos + wq0 : -1, wave_last = mine ? min(a.pos + wq0 + 15, tile.len - 1) : -1;  // last position any query of the wave sees
  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;

  uint4 qf[NK];
  int qpos;
  load_queries<D>(qf, qpos, a, sq, h, mine ? wq0 + m : sq.S, g);
  f32x4 o[ND];
  float m_run, l_run;
  flow_walk<D, true>(tile, first, end, wave, qf, qpos, wave_first, wave_last, lds0, a.scale_log2e, o, m_run, l_run);
  if (!mine) return;
  l_run = lane_xor_sum<32>(lane_xor_sum<16>(l_run));
  float* part = c.part + ((size_t)(bh * c.cut.tasks + task) * c.cut.chunks + chunk) * PS;
#pragma unroll
  for (int db = 0; db < ND; ++db) *reinterpret_cast<f32x4*>(part + (db * 64 + lane) * 4) = o[db];
  if (g == 0) {
    part[16 * D + m] = m_run;
    part[16 * D + 16 + m] = l_run;
  }
}

// The chunks' sums of a task, in their order: a wave takes sixteen columns of its sixteen queries.
template <int D, bool FEW>
__global__ __launch_bounds__(D * 4) void attn_chunks_merge_kernel(ChunkArgs c) {
  constexpr int PS = 16 * D + 32;
  const PrefillArgs& a = c.p;
  const int lane = threadIdx.x & 63, db = threadIdx.x >> 6, m = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x / c.cut.tasks, task = blockIdx.x - bh * c.cut.tasks, b = bh / a.Hkv;
  const int qi = task / c.group * 16 + m, h = (bh - b * a.Hkv) * c.group + task % c.group;
  const float* part = c.part + (size_t)blockIdx.x * c.cut.chunks * PS;
  float M = -INFINITY, l = 0.f;
  f32x4 sum = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < c.cut.chunks; i0 += 8) {  // eight chunks' loads in flight; the maxima are whole powers of two, so is every rescaling
    float mx[8], ls[8];
    f32x4 pv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float* p = part + (size_t)min(i0 + i, c.cut.chunks - 1) * PS;
      mx[i] = i0 + i < c.cut.chunks ? p[16 * D + m] : -INFINITY;
      ls[i] = p[16 * D + 16 + m];
      pv[i] = *reinterpret_cast<const f32x4*>(p + (db * 64 + lane) * 4);
    }
    float mn = M;
#pragma unroll
    for (int i = 0; i < 8; ++i) mn = fmaxf(mn, mx[i]);
    const float back = pow2_neg_int(M - mn);
    l *= back;
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[e] *= back;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float w = mx[i] == -INFINITY ? 0.f : pow2_neg_int(mx[i] - mn);
      l += ls[i] * w;
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = i0 + i < c.cut.chunks ? __builtin_fmaf(pv[i][e], w, sum[e]) : sum[e];  // (an infinity: not twice)
    }
    M = mn;
  }
  const unsigned int odd = FEW ? columns_not_finite((sum[0] + sum[1]) + (sum[2] + sum[3])) : 0;
  if (qi < a.S && !(odd >> m & 1)) {
    const float inv = 1.0f / l;
    *reinterpret_cast<uint2*>(a.out + ((size_t)b * a.S + qi) * a.H * D + (size_t)h * D + 16 * db + 4 * g) =
        make_uint2(pack_bf(sum[0] * inv, sum[1] * inv), pack_bf(sum[2] * inv, sum[3] * inv));
  }
  if (FEW && odd) walk_rows<D>(a, sequence(a, b), h, 0, odd, 16 * db, 16, lane);
}

// How a call would be cut: no chunks (0) where the kernels above are the better ones, which is where the walk is no longer than 512
// positions and two more for every task (the more tasks, the more CUs they keep, and the more partial sums).  us, uncut / cut:
//   16 x 6 heads behind 500    9.1 /  8.2  (not cut)     8 x 24 x 16 (4) behind 1000 14.5 / 14.7  (not cut)
//   behind 1000               13.6 /  8.4                8 x 48 x 16 (4) behind 1000 18.2 / 18.5  (not cut)
//   2 x 128 x 16 (4), 400      9.5 / 12.2  (not cut)     8 x 100 x 6 behind 3000     44.8 / 26.2
//   1024 x 6 from the start   16.7 / 18.3  (not cut)     8 x 100 x 16 (4) behind 3000 66.6 / 45.7
// A workgroup a CU, so as not to write more partial sums than that takes (48 a KV head: 4 x 48 x 16 (4) behind 1900 17.3 us, with two a
// CU 18.3); two from 65 on, where one leaves CUs idle (96: 8 x 100 x 6 39.7, with two 26.2).  None under three tiles.
// One or two tasks over many KV heads read their positions at the rate of HBM as they are: 16 queries behind 1500, 192 heads of 128 25.7 /
// 28.2, 128 22.5 / 23.0, but 32 queries and 96 heads 20.9 / 19.6; 192 heads of 64 17.4 / 18.4, but 144 16.6 / 14.8.
inline Cut cut(int B, int S, int H, int Hkv, int D, int pos, bool most = false) {  // most: the chunks of any call at `pos` or before
  constexpr int CUS = 256;
  const int64_t tasks = (int64_t)((S + 15) / 16) * (H / Hkv), ntb = (tasks + 3) / 4, wgs = ntb * B * Hkv;
  const int ntiles = (int)((pos + (int64_t)S + KT - 1) / KT);
  if (wgs > CUS || pos + (int64_t)S <= 512 + 2 * tasks * B * Hkv) return Cut{};
  if (tasks < 3 && (int64_t)B * Hkv > (D == 128 ? 112 : 160)) return Cut{};
  const int want = (int)((wgs <= 64 ? CUS : 2 * CUS) / wgs);
  const int tiles = std::max((ntiles + want - 1) / want, 3);
  return Cut{(int)tasks, (int)ntb, most ? std::min(want, (ntiles + 2) / 3) : (ntiles + tiles - 1) / tiles, tiles};
}

template <int D>
int launch_chunks(const PrefillArgs& a, const Cut& cut, float* part, hipStream_t st) {
  const ChunkArgs c{a, cut, a.H / a.Hkv, part};
  const int n = c.p.B * c.p.Hkv * c.cut.ntb * c.cut.chunks;
  hipLaunchKernelGGL((attn_chunk_kernel<D>), dim3((n + 7) / 8 * 8), dim3(256), 2 * KvTile<D>::SLOT, st, c);
  const dim3 tasks(c.p.B * c.p.Hkv * c.cut.tasks);
  if (a.S < 16) hipLaunchKernelGGL((attn_chunks_merge_kernel<D, true>), tasks, dim3(D * 4), 0, st, c);
  else hipLaunchKernelGGL((attn_chunks_merge_kernel<D, false>), tasks, dim3(D * 4), 0, st, c);
  return ohara_launch_status();
}

template <int D, int QW, bool ALIGNED = true, bool FEW = false>
int launch_waves(PrefillArgs a, hipStream_t st) {
  a.nqb = (a.S + 64 * QW - 1) / (64 * QW);
  const int64_t blocks = a.nqb * (a.seqs ? ((int64_t)a.H * a.B + 7) / 8 * 8 : (int64_t)a.H * a.B);
  if (blocks > INT32_MAX) return OHARA_ESIZE;
  hipLaunchKernelGGL((attn_prefill_kernel<D, QW, ALIGNED, FEW>), dim3((unsigned)blocks), dim3(256), 2 * KvTile<D>::SLOT, st, a);
  return ohara_launch_status();
}

template <int D>
int launch_flow(PrefillArgs a, hipStream_t st) {
  a.nqb = (a.S + 63) / 64;
  const int64_t blocks = a.nqb * (a.seqs ? ((int64_t)a.H * a.B + 7) / 8 * 8 : (int64_t)a.H * a.B);
  if (blocks > INT32_MAX) return OHARA_ESIZE;
  hipLaunchKernelGGL((attn_flow_kernel<D>), dim3((unsigned)blocks), dim3(256), 2 * KvTile<D>::SLOT, st, a);
  return ohara_launch_status();
}

template <int D, int TEAMS, bool FEW = false, int NST = 3>
int launch_teams(PrefillArgs a, hipStream_t st) {
  constexpr int LDS = NST * KvTile<D>::SLOT + 2 * TEAMS * 4096;
  a.nqb = (a.S + 16 * TEAMS - 1) / (16 * TEAMS);
  if (LDS > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)attn_team_kernel<D, TEAMS, NST, true, FEW>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  hipLaunchKernelGGL((attn_team_kernel<D, TEAMS, NST, true, FEW>), dim3((unsigned)(a.nqb * (a.seqs ? (a.H * a.B + 7) / 8 * 8 : a.H * a.B))), dim3(TEAMS * 256), LDS, st, a);
  return ohara_launch_status();
}

// All kernels give the same bits; us with teams of 16 / 32 queries a workgroup and attn_prefill_kernel's waves of 16 / 32 (64 / 128 a workgroup):
//   heads of 128                                                 heads of 64, 16 heads
//     128 queries x 6 heads   4.5 /  5.5 /  5.5 /  7.1             160 queries      4.3 /  5.0 /  4.6 /  5.8
//     48 behind 1900, 4 x 16 24.7 / 27.8 / 34   / 49               500              7.6 /  8.5 /  8.4 / 11.7
//     600 x 6                10.4 / 11.4 / 13.0 / 18.6             24 x 160         23  / 18   /  9.8 /  9.9
//     1024 x 6               22   / 16.7 / 20   / 28               8 x 1024         122 / 90   / 34.9 / 36.1
//     1024 x 16              31   / 20.3 / 20.2 / 28
//     4001 x 16             364   / 214  / 110  / 122
//     8 x 1024 x 6           97   / 62   / 28   / 36
//     32 x 512 x 6          137   / 84   / 38   / 31
//     16 x 700 x 16         269   / 173  / 74   / 68
// so: teams of 16 while every one has a CU to itself, and over more than two tiles while every two have one (with heads of 128
// as teams of 32).  A shorter walk does not pay for the teams' barriers: us, teams / waves: heads of 64, 8 x 24 queries x 32 heads
// 5.2 / 4.8; heads of 128, 8 x 33 x 16 6.2 / 5.4; over four tiles, 200 x 32 7.1 / 7.5.
// The rest is drawn through 384 calls of 65 to 4096 tokens, 1 to 64 sequences, five combinations of heads of 64 and of 128, behind 0 to 2000: within
// 1 % of the best of the three on average (29 % at worst), and 6 % quicker than attn_prefill_kernel alone.  us, its 16 / its 32 queries a wave /
// attn_flow_kernel (16):
// * 128 queries a workgroup read each position once where 64 read it twice, and are slower by a quarter where there are few of them or the second half of
//   the last one is empty.  So from three a CU on, if at least half of their second halves hold queries (heads of 128: 16 x 468 x 16 behind 1000 160 / 122 /
//   170, 8 x 512 x 16 26.7 / 26.7 / 25.8, 4 x 1073 x 16 behind 1500 156 / 131 / 117); with heads of 64 also from the sixth workgroup of 64 queries a
//   CU (32 x 65 x 32 behind 1500 168 / 111 / 154; four, 8 x 512 x 16 14.8 / 18.1 / 16.9); with heads of 128 from the second of 128 if a sequence is one of
//   them: all of one length (32 x 90 x 16 behind 1000 108 / 69 / 105, 16 x 100 x 32 18.5 / 15.8 / 18.3, 48 x 65 x 6 behind 1500 97 / 79 / 78).
// * Else attn_flow_kernel (4001 x 6 heads of 128 behind 500 70 / 93 / 53, 8 x 65 x 16 behind 1000 35 / 44 / 26), but not over two tiles at most, which leaves
//   little to overlap (12 x 100 x 16 9.4 / 9.8 of 16 queries), nor over a short walk where its workgroups, two a CU, need a second round: heads of 128, 8 x 300 x 16
//   15.3 / 16.9 / 16.5, 4 x 383 x 32 19.6 / 21.1 / 20.6; heads of 64, of which the other has four a CU, 4 x 512 x 32 14.4 / 17.5 / 16.5, 16 x 128 x 32
//   behind 37 11.4 / 12.5 / 13.5, and over walks of one length 16 x 94 x 32 behind 2000 78 / 82 / 89, 8 x 640 x 12 behind 1500 53 / 61 / 56 (of many
//   lengths, 2 x 4045 x 8 from the start 66 / 85 / 54).
template <int D>
int launch_prefill_for(const PrefillArgs& a, const int32_t* lengths, hipStream_t st) {  // lengths: on the host, where they differ
  constexpr int CUS = 256;
  auto blocks = [&](int queries) {
    if (!lengths) return (a.S + queries - 1) / queries * (int64_t)a.H * a.B;
    int64_t n = 0;
    for (int b = 0; b < a.B; ++b) n += (lengths[b] + queries - 1) / queries;
    return n * a.H;
  };
  const bool aligned = !(((uintptr_t)a.k | (uintptr_t)a.v) & 15), long_walk = a.pos + a.S > 128;
  if (a.S < 16 && !a.seqs) {  // (a call's own tokens; the rules below come to the same kernels)
    if (!aligned) return launch_waves<D, 1, false, true>(a, st);
    return blocks(16) <= CUS * (D == 64 && long_walk ? 2 : 1) ? launch_teams<D, 1, true>(a, st) : launch_waves<D, 1, true, true>(a, st);
  }
  if (!aligned) return launch_waves<D, 1, false>(a, st);
  if (blocks(16) <= CUS * (D == 64 && long_walk ? 2 : 1)) return launch_teams<D, 1>(a, st);
  if constexpr (D == 128)
    if (long_walk && blocks(32) <= CUS) return launch_teams<D, 2>(a, st);
  const int64_t wide = blocks(128), halves = blocks(64);
  const bool two_a_cu = D == 64 ? halves > 5 * CUS : wide > CUS && a.S <= 128;
  if ((wide >= 3 * CUS || two_a_cu) && 2 * halves >= 3 * wide) return launch_waves<D, 2>(a, st);
  const int far = a.pos + a.S;
  const bool second_round = D == 128 ? halves > 2 * CUS && halves <= 3 * CUS && far <= 512
                                     : (halves > 11 * CUS / 4 && halves <= 17 * CUS / 4 && far < 1000) ||
                                           (halves > 13 * CUS / 4 && halves <= 4 * CUS && a.pos + 64 >= a.S);
  return long_walk && !second_round ? launch_flow<D>(a, st) : launch_waves<D, 1>(a, st);
}

}  // namespace

static int prefill_args(PrefillArgs& a, const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch, int seq_len, int h, int h_kv,
                        int dh, int t_max, int pos, uint16_t* out) {
  if (!q || !kcache || !vcache || !out) return OHARA_EINVAL;
  if (batch < 1 || seq_len < 1 || h < 1 || h_kv < 1 || h % h_kv || t_max < 1) return OHARA_EINVAL;
  if (pos < 0 || pos + seq_len > t_max) return OHARA_EINVAL;
  if (dh != 64 && dh != 128) return OHARA_ESIZE;
  if (batch > 65535 || h > 65535) return OHARA_ESIZE;
  a.q = q; a.k = kcache; a.v = vcache; a.out = out;
  a.B = batch; a.S = seq_len; a.H = h; a.Hkv = h_kv; a.Tmax = t_max; a.pos = pos;
  a.scale_log2e = (1.0f / sqrtf((float)dh)) * OHARA_LOG2E;  // the same constant as the decode kernels'
  return OHARA_OK;
}

extern "C" int ohara_attn_prefill_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch,
                                       int seq_len, int h, int h_kv, int dh, int t_max, int pos, uint16_t* out,
                                       void* stream) {
  PrefillArgs a{};
  const int rc = prefill_args(a, q, kcache, vcache, batch, seq_len, h, h_kv, dh, t_max, pos, out);
  if (rc) return rc;
  return dh == 128 ? launch_prefill_for<128>(a, nullptr, (hipStream_t)stream) : launch_prefill_for<64>(a, nullptr, (hipStream_t)stream);
}

// The partial results of a call that is cut into chunks: task x chunk blocks of 16 dh sums and 32 statistics.
static int64_t chunk_bytes(const Cut& c, int batch, int h_kv, int dh) {
  return (int64_t)batch * h_kv * c.tasks * c.chunks * (16 * dh + 32) * (int64_t)sizeof(float);
}

extern "C" int64_t ohara_attn_prefill_ws_bytes(int batch, int seq_len, int h, int h_kv, int dh, int pos) {
  if (batch < 1 || seq_len < 1 || h < 1 || h_kv < 1 || h % h_kv || (dh != 64 && dh != 128) || pos < 0) return OHARA_EINVAL;
  return chunk_bytes(cut(batch, seq_len, h, h_kv, dh, pos, true), batch, h_kv, dh);
}

// Two to fifteen tokens a sequence: ohara_attn_cached_bf16 walks the context once for every token, in a workgroup of its own; the same
// products, weights rounded the same way.  us, it / these:
//   heads of 128, each with its keys, 6 heads                            16 heads
//     2 behind 500            5.9 /  8.2   4 x 4 behind 500 10.9 /  8.2   8 behind 200       4.8 /  5.8   8 x 2 behind 200     7.5 /  5.7
//     2 behind 1000           8.8 /  8.4   8 x 4 behind 200  6.6 /  5.8   4 behind 500      11.1 /  8.3   8 x 8 behind 30      6.7 /  4.0
//     8 behind 3000            49 /  9.7   8 x 15 behind 3000 184 / 21.3   2 x 4 behind 200   5.4 /  5.7   8 x 15 behind 3000   459 / 40.7
//   16 heads of 64: 2 x 8 behind 200 4.2 / 4.9; 4 x 8 8.8 / 4.9; 8 x 2 behind 500 9.1 / 6.9; 2 x 2 5.0 / 6.8
//   16 heads of 128 on 4 of keys: 2 behind 30 4.7 / 3.8; 8 behind 3000 55 / 10.7; 8 x 15 124 / 18.5
// (2 behind 1000 in one walk, without room: 13.6 us)
extern "C" int ohara_attn_prefill_wins_with(int batch, int seq_len, int h, int h_kv, int dh, int pos, int64_t workspace_bytes) {
  if (batch < 1 || seq_len < 2 || h < 1 || h_kv < 1 || h % h_kv || (dh != 64 && dh != 128) || pos < 0) return 0;
  if (seq_len >= 16) return 1;
  if (batch > 65535 || h > 65535) return 0;
  const int64_t walks = (int64_t)batch * seq_len * h_kv, far = (int64_t)pos + seq_len;
  const Cut c = cut(batch, seq_len, h, h_kv, dh, pos);
  return h / h_kv > 2 || (c.chunks > 1 && workspace_bytes >= chunk_bytes(c, batch, h_kv, dh)) || walks >= 512 ||
         (walks >= 256 * 128 / dh && far >= 128) || (walks >= 96 && far >= 384);
}

extern "C" int ohara_attn_prefill_wins(int batch, int seq_len, int h, int h_kv, int dh, int pos) {
  return ohara_attn_prefill_wins_with(batch, seq_len, h, h_kv, dh, pos, INT64_MAX);
}

extern "C" int ohara_attn_prefill_ws_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch, int seq_len, int h,
                                          int h_kv, int dh, int t_max, int pos, uint16_t* out, void* workspace, int64_t workspace_bytes,
                                          void* stream) {
  PrefillArgs a{};
  const int rc = prefill_args(a, q, kcache, vcache, batch, seq_len, h, h_kv, dh, t_max, pos, out);
  if (rc) return rc;
  const hipStream_t st = (hipStream_t)stream;
  const Cut c = cut(batch, seq_len, h, h_kv, dh, pos);
  if (c.chunks > 1 && workspace && workspace_bytes >= chunk_bytes(c, batch, h_kv, dh) &&
      !(((uintptr_t)workspace | (uintptr_t)kcache | (uintptr_t)vcache) & 15))
    return dh == 128 ? launch_chunks<128>(a, c, (float*)workspace, st) : launch_chunks<64>(a, c, (float*)workspace, st);
  return dh == 128 ? launch_prefill_for<128>(a, nullptr, st) : launch_prefill_for<64>(a, nullptr, st);
}

extern "C" int ohara_attn_prompts_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int n, const int32_t* lengths,
                                       const int32_t* seqs, int h, int h_kv, int dh, int t_max, uint16_t* out, void* stream) {
  if (!q || !kcache || !vcache || !lengths || !seqs || !out) return OHARA_EINVAL;
  if (n < 1 || h < 1 || h_kv < 1 || h % h_kv || t_max < 1) return OHARA_EINVAL;
  if (dh != 64 && dh != 128) return OHARA_ESIZE;
  if (n > 65535 || h > 65535) return OHARA_ESIZE;
  PrefillArgs a{};
  a.q = q; a.k = kcache; a.v = vcache; a.out = out; a.seqs = seqs;
  a.B = n; a.H = h; a.Hkv = h_kv; a.Tmax = t_max;
  for (int b = 0; b < n; ++b) {
    if (lengths[b] < 1 || lengths[b] > t_max) return OHARA_EINVAL;
    if (lengths[b] > a.S) a.S = lengths[b];
  }
  a.scale_log2e = (1.0f / sqrtf((float)dh)) * OHARA_LOG2E;
  return dh == 128 ? launch_prefill_for<128>(a, lengths, (hipStream_t)stream) : launch_prefill_for<64>(a, lengths, (hipStream_t)stream);
}
