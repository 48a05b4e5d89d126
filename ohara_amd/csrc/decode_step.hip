// Llama.forward through the KV cache (ohara/models/llama.py:279-323) as a fixed chain
// of five kernels per layer:
//   norm1 + QKV projection + rotary + cache append     (Block :199, Attention :84-98)
//   attention over the cache                           (:100-135)
//   output projection + residual                       (:142, :199)
//   norm2 + gate/up projection + SwiGLU                (:200, mlp.py:152)
//   down projection + residual                         (:200)
// then final norm + vocabulary projection (:321-322) and, optionally, greedy
// selection feeding the next step.  No host synchronisation, no allocation: the
// chain can be captured once into a HIP graph and replayed per token.
#include "gemm_epilogue.h"

#include <algorithm>
#include <type_traits>
#include <utility>

extern "C" int ohara_llama_forward(const OharaModel* m, const OharaDecodeState* s, int seq_len, int pos,
                                   int use_pos_dev, int logits_mode, int select_greedy, void* stream) {
  if (!m || !s || !m->layers || !s->kcache || !s->vcache) return OHARA_EINVAL;
  if (s->kv_int8 && (!s->kvstats || !s->kstage || !s->vstage)) return OHARA_EINVAL;
  if (s->batch < 1 || seq_len < 1) return OHARA_EINVAL;
  const int64_t rows64 = (int64_t)s->batch * seq_len;
  if (rows64 > s->rows_cap) return OHARA_ESIZE;
  const bool ragged = s->seq_pos != nullptr;
  if (!ragged && use_pos_dev && (!s->step_state || seq_len != 1)) return OHARA_EINVAL;
  if (!ragged && !use_pos_dev && (pos < 0 || pos + seq_len > m->t_max)) return OHARA_EINVAL;
  if (logits_mode < OHARA_LOGITS_NONE || logits_mode > OHARA_LOGITS_ALL) return OHARA_EINVAL;
  if (select_greedy && !(logits_mode == OHARA_LOGITS_LAST || (logits_mode == OHARA_LOGITS_ALL && seq_len == 1)))
    return OHARA_EINVAL;
  const int B = s->batch, R = (int)rows64;
  const int d = m->d_model, H = m->n_heads, Hkv = m->n_kv_heads, Dh = m->head_dim;
  const int32_t* pos_dev = use_pos_dev ? s->step_state : nullptr;  // first field is pos
  const int n_split = seq_len == 1 ? s->n_split : 1;
  hipStream_t hs = (hipStream_t)stream;
  // of attn_ws, what lies behind the counters of decode attention (which stay zero) is room for a prompt's partial results
  const int64_t counters = ((int64_t)B * Hkv * 4 + 255) / 256 * 256;
  const int64_t room = s->attn_ws && !((uintptr_t)s->attn_ws & 15) ? std::max<int64_t>(0, ohara_attn_workspace_bytes(B, H, Hkv, Dh, s->n_split) - counters) : 0;
  void* const room_at = s->attn_ws ? (unsigned char*)s->attn_ws + counters : nullptr;
  int launch = 0;
  // Brackets launch number s->prof_kernel with the caller's events.
#define OHARA_RUN(call)                                                                     \
  do {                                                                                      \
    const bool prof_ = (launch == s->prof_kernel) && s->prof_start && s->prof_stop;         \
    if (prof_) (void)hipEventRecord((hipEvent_t)s->prof_start, hs);                         \
    rc = (call);                                                                            \
    if (prof_) (void)hipEventRecord((hipEvent_t)s->prof_stop, hs);                          \
    ++launch;                                                                               \
    if (rc) return rc;                                                                      \
  } while (0)
  int rc = 0;
  // many rows: normed once, then the tiled MFMA kernel (launches are not numbered)
  auto normed = [&](int n) { return s->xn != nullptr && ohara_norm_ahead(R, d, (n + 15) / 16 * 16); };
  const bool qkv_normed = normed((H + 2 * Hkv) * Dh), gu_normed = normed(2 * ((m->d_ff + 7) / 8 * 8));
  const bool logits_normed = logits_mode == OHARA_LOGITS_ALL && normed(m->vocab);
  OHARA_RUN(ohara_embed_bf16(s->ids, m->token_emb, s->x, R, d, m->vocab, stream));
  for (int l = 0; l < m->n_layers; ++l) {
    const OharaLayer& L = m->layers[l];
    if (qkv_normed && l == 0) {  // later layers' norms come with the residual before them
      rc = ohara_rmsnorm_bf16(s->x, L.norm1, s->xn, R, d, m->eps, stream);
      if (rc) return rc;
    }
    if (ragged && s->kv_int8) {
      // one position per sequence over the int8 cache: rows to staging, quantise into the cache at each sequence's
      // own position, attention straight over the codes (the extra launch is not numbered)
      int8_t* kq = reinterpret_cast<int8_t*>(s->kcache[l]);
      int8_t* vq = reinterpret_cast<int8_t*>(s->vcache[l]);
      OHARA_RUN(ohara_qkv_rope_ragged_bf16(qkv_normed ? s->xn : s->x, d, L.wqkv, d, qkv_normed ? nullptr : L.norm1, m->eps, B,
                                           seq_len, H, Hkv, Dh, m->cos, m->sin, s->seq_pos, m->t_max, s->q, s->kstage,
                                           s->vstage, stream));
      if (seq_len == 1) {
        OHARA_RUN(ohara_attn_append_int8(s->q, s->kstage, s->vstage, kq, vq, s->kvstats[l], B, H, Hkv, Dh, m->t_max, 0, s->seq_pos, 1,
                                         n_split, s->attn_ws, s->attn, stream));
      } else {
        rc = ohara_kv_quant_append_ragged_int8(s->kstage, s->vstage, B, seq_len, Hkv, Dh, s->seq_pos, kq, vq, s->kvstats[l],
                                               m->t_max, stream);
        if (rc) return rc;
        OHARA_RUN(ohara_attn_cached_ragged_int8(s->q, kq, vq, s->kvstats[l], B, seq_len, H, Hkv, Dh, m->t_max, s->seq_pos,
                                                n_split, s->attn_ws, s->attn, stream));
      }
    } else if (ragged) {
      // one position per sequence; attention of any length through the split-context kernel
      OHARA_RUN(ohara_qkv_rope_append_ragged_bf16(qkv_normed ? s->xn : s->x, d, L.wqkv, d, qkv_normed ? nullptr : L.norm1, m->eps,
                                                  B, seq_len, H, Hkv, Dh, m->cos, m->sin, s->seq_pos, s->q, s->kcache[l],
                                                  s->vcache[l], m->t_max, stream));
      OHARA_RUN(ohara_attn_cached_ragged_bf16(s->q, s->kcache[l], s->vcache[l], B, seq_len, H, Hkv, Dh, m->t_max,
                                              s->seq_pos, n_split, s->attn_ws, s->attn, stream));
    } else if (!s->kv_int8) {
      OHARA_RUN(ohara_qkv_rope_append_bf16(qkv_normed ? s->xn : s->x, d, L.wqkv, d, qkv_normed ? nullptr : L.norm1, m->eps, B,
                                           seq_len, H, Hkv, Dh, m->cos, m->sin, pos, pos_dev, s->q, s->kcache[l],
                                           s->vcache[l], m->t_max, stream));
      if (ohara_attn_prefill_wins_with(B, seq_len, H, Hkv, Dh, pos, room))
        OHARA_RUN(ohara_attn_prefill_ws_bf16(s->q, s->kcache[l], s->vcache[l], B, seq_len, H, Hkv, Dh, m->t_max, pos,
                                             s->attn, room_at, room, stream));
      else
        OHARA_RUN(ohara_attn_cached_bf16(s->q, s->kcache[l], s->vcache[l], B, seq_len, H, Hkv, Dh, m->t_max, pos,
                                         pos_dev, n_split, s->attn_ws, s->attn, stream));
    } else {
      // int8 cache (kv_cache.py:94-102): rows to staging, quantise into the cache, attention on the
      // dequantised values (the extra launches are not numbered)
      int8_t* kq = reinterpret_cast<int8_t*>(s->kcache[l]);
      int8_t* vq = reinterpret_cast<int8_t*>(s->vcache[l]);
      OHARA_RUN(ohara_qkv_rope_bf16(qkv_normed ? s->xn : s->x, d, L.wqkv, d, qkv_normed ? nullptr : L.norm1, m->eps, B, seq_len, H,
                                    Hkv, Dh, m->cos, m->sin, pos, pos_dev, m->t_max, s->q, s->kstage, s->vstage, stream));
      if (seq_len > 1) {
        rc = ohara_kv_quant_append_int8(s->kstage, s->vstage, B, seq_len, Hkv, Dh, pos, pos_dev, kq, vq, s->kvstats[l],
                                        m->t_max, stream);
        if (rc) return rc;
      }
      if (seq_len == 1) {
        OHARA_RUN(ohara_attn_append_int8(s->q, s->kstage, s->vstage, kq, vq, s->kvstats[l], B, H, Hkv, Dh, m->t_max, pos, pos_dev, 0,
                                         n_split, s->attn_ws, s->attn, stream));
      } else if (seq_len >= 16 && (Dh == 64 || Dh == 128) && s->kdeq && s->vdeq) {
        const int len = pos + seq_len;
        rc = ohara_kv_dequant_int8(kq, s->kvstats[l], 0, B, len, Hkv, Dh, m->t_max, s->kdeq, stream);
        if (!rc) rc = ohara_kv_dequant_int8(vq, s->kvstats[l], 1, B, len, Hkv, Dh, m->t_max, s->vdeq, stream);
        if (rc) return rc;
        OHARA_RUN(ohara_attn_prefill_ws_bf16(s->q, s->kdeq, s->vdeq, B, seq_len, H, Hkv, Dh, len, pos, s->attn, room_at, room, stream));
      } else {
        OHARA_RUN(ohara_attn_cached_int8(s->q, kq, vq, s->kvstats[l], B, seq_len, H, Hkv, Dh, m->t_max, pos, pos_dev,
                                         n_split, s->attn_ws, s->attn, stream));
      }
    }
    const bool parts = qkv_normed || gu_normed;
    if (parts)
      OHARA_RUN(ohara_gemm_residual_norm_bf16(s->attn, H * Dh, L.wo, d, H * Dh, R, s->x, gu_normed ? L.norm2 : nullptr, m->eps, s->xn, room_at,
                                              room, stream));
    else
      OHARA_RUN(ohara_gemm_skinny_bf16(s->attn, H * Dh, L.wo, d, H * Dh, nullptr, m->eps, R, OHARA_EPI_RESIDUAL, s->x, d, s->x, d, stream));
    OHARA_RUN(ohara_gemm_skinny_bf16(gu_normed ? s->xn : s->x, d, L.wgu, m->d_ff, d, gu_normed ? nullptr : L.norm2, m->eps, R,
                                     OHARA_EPI_SWIGLU, nullptr, 0, s->act, m->d_ff, stream));
    const bool last = l + 1 == m->n_layers;
    const uint16_t* after = last ? (logits_normed ? m->final_norm : nullptr) : qkv_normed ? m->layers[l + 1].norm1 : nullptr;
    if (parts || after)
      OHARA_RUN(ohara_gemm_residual_norm_bf16(s->act, m->d_ff, L.wdown, d, m->d_ff, R, s->x, after, m->eps, s->xn, room_at, room, stream));
    else
      OHARA_RUN(ohara_gemm_skinny_bf16(s->act, m->d_ff, L.wdown, d, m->d_ff, nullptr, m->eps, R, OHARA_EPI_RESIDUAL, s->x, d, s->x, d, stream));
  }
  if (logits_mode == OHARA_LOGITS_ALL) {
    OHARA_RUN(ohara_gemm_skinny_bf16(logits_normed ? s->xn : s->x, d, m->w_vocab, m->vocab, d, logits_normed ? nullptr : m->final_norm,
                                     m->eps, R, OHARA_EPI_STORE, nullptr, 0, s->logits, m->vocab, stream));
  } else if (logits_mode == OHARA_LOGITS_LAST) {
    // row b*seq_len + seq_len-1 of x for every sequence: a strided view, no gather
    OHARA_RUN(ohara_gemm_skinny_bf16(s->x + (size_t)(seq_len - 1) * d, seq_len * d, m->w_vocab, m->vocab, d,
                                     m->final_norm, m->eps, B, OHARA_EPI_STORE, nullptr, 0, s->logits, m->vocab,
                                     stream));
  }
  if (select_greedy)
    OHARA_RUN(ohara_argmax_bf16(s->logits, m->vocab, B, m->vocab, s->valid_vocab > 0 ? s->valid_vocab : m->vocab,
                                s->ids, s->history, s->hist_cap, s->step_state, stream));
#undef OHARA_RUN
  return OHARA_OK;
}

// The last row of every prompt, 16 bytes a lane.
static __global__ __launch_bounds__(64) void last_rows_kernel(const bf16_t* x, const int32_t* seqs, bf16_t* out, int d) {
  const int b = blockIdx.x, n = gridDim.x;
  const size_t row = (size_t)seqs[b] + seqs[n + b] - 1;
  for (int i = threadIdx.x * 8; i < d; i += 512) *reinterpret_cast<uint4*>(out + (size_t)b * d + i) = ldg16(x + row * d + i);
}

// The same chain over prompts of different lengths, each from position 0 into its own row of the caches: the row-wise kernels
// run once over all rows, side by side without padding.  16 prompts of 100 to 800 tokens, d12: 11.8 ms one by one, 4.1 together.
extern "C" int ohara_llama_prompts(const OharaModel* m, const OharaDecodeState* s, int n, const int32_t* lengths, const int32_t* table,
                                   void* stream) {
  if (!m || !s || !m->layers || !s->kcache || !s->vcache || !lengths || !table || !s->xn || !s->logits) return OHARA_EINVAL;
  if (s->kv_int8 || n < 1) return OHARA_EINVAL;
  int64_t rows = 0;
  for (int b = 0; b < n; ++b) {
    if (lengths[b] < 1 || lengths[b] > m->t_max) return OHARA_EINVAL;
    rows += lengths[b];
  }
  if (rows > s->rows_cap) return OHARA_ESIZE;
  const int R = (int)rows, d = m->d_model, H = m->n_heads, Hkv = m->n_kv_heads, Dh = m->head_dim;
  if (d & 7) return OHARA_ESIZE;
  const int32_t* at = table + 3 * n;
  int rc = ohara_embed_bf16(s->ids, m->token_emb, s->x, R, d, m->vocab, stream);
  for (int l = 0; l < m->n_layers && !rc; ++l) {
    const OharaLayer& L = m->layers[l];
    rc = ohara_rmsnorm_bf16(s->x, L.norm1, s->xn, R, d, m->eps, stream);
    if (!rc) rc = ohara_qkv_rope_append_rows_bf16(s->xn, d, L.wqkv, d, R, H, Hkv, Dh, m->cos, m->sin, at, s->q, s->kcache[l],
                                                  s->vcache[l], m->t_max, stream);
    if (!rc) rc = ohara_attn_prompts_bf16(s->q, s->kcache[l], s->vcache[l], n, lengths, table, H, Hkv, Dh, m->t_max, s->attn, stream);
    if (!rc) rc = ohara_gemm_bf16(s->attn, H * Dh, L.wo, d, H * Dh, R, OHARA_EPI_RESIDUAL, s->x, d, s->x, d, stream);
    if (!rc) rc = ohara_rmsnorm_bf16(s->x, L.norm2, s->xn, R, d, m->eps, stream);
    if (!rc) rc = ohara_gemm_bf16(s->xn, d, L.wgu, m->d_ff, d, R, OHARA_EPI_SWIGLU, nullptr, 0, s->act, m->d_ff, stream);
    if (!rc) rc = ohara_gemm_bf16(s->act, m->d_ff, L.wdown, d, m->d_ff, R, OHARA_EPI_RESIDUAL, s->x, d, s->x, d, stream);
  }
  if (rc) return rc;
  hipLaunchKernelGGL(last_rows_kernel, dim3(n), dim3(64), 0, (hipStream_t)stream, s->x, table, s->xn, d);
  return ohara_gemm_skinny_bf16(s->xn, d, m->w_vocab, m->vocab, d, m->final_norm, m->eps, n, OHARA_EPI_STORE, nullptr, 0, s->logits,
                                m->vocab, stream);
}

extern "C" int ohara_event_create(void** event) {
  if (!event) return OHARA_EINVAL;
  hipEvent_t e;
  if (hipEventCreate(&e) != hipSuccess) return OHARA_ELAUNCH;
  *event = e;
  return OHARA_OK;
}
extern "C" int ohara_event_destroy(void* event) {
  return hipEventDestroy((hipEvent_t)event) == hipSuccess ? OHARA_OK : OHARA_ELAUNCH;
}
extern "C" int ohara_event_record(void* event, void* stream) {
  return hipEventRecord((hipEvent_t)event, (hipStream_t)stream) == hipSuccess ? OHARA_OK : OHARA_ELAUNCH;
}
extern "C" int ohara_event_elapsed_ms(void* start, void* stop, float* ms) {
  if (!ms) return OHARA_EINVAL;
  return hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop) == hipSuccess ? OHARA_OK : OHARA_ELAUNCH;
}

// The chain over experts.  A step of one sequence through 16 layers of 64 experts was bound by the host, nine calls of Python a layer:
// 1.19 ms, from here 0.74 (4 sequences 1.18 / 0.85; from 16 on it is the kernels either way).
namespace {

struct MoeScratch {
  uint16_t *x, *y, *xn, *q, *attn, *k, *v, *kd, *vd, *w, *act, *act_sh, *out, *router;
  int32_t *idx, *meta;
  void* room;
  int64_t room_bytes, bytes;
  bool attend_rows, dequantise;  // attention by the prompt kernels; over a bfloat16 copy of an int8 cache
};

// What a call keeps where; false where it is not one that this chain takes.
bool moe_scratch(const OharaMoeCall& c, MoeScratch& s) {
  if (c.n_layers < 1 || c.batch < 1 || c.seq_len < 1 || c.pos < 0 || c.t_max < 1 || c.pos > c.t_max - c.seq_len || c.n_split < 1) return false;
  if (c.d_model < 8 || c.n_heads < 1 || c.n_kv_heads < 1 || c.n_heads % c.n_kv_heads || c.head_dim < 2 || c.vocab < 1 || !c.layers) return false;
  const int64_t R = (int64_t)c.batch * c.seq_len, d = c.d_model;
  if (R > (1 << 20)) return false;
  int64_t act = 0, act_sh = 0, pairs = 0, experts = 0;
  for (int l = 0; l < c.n_layers; ++l) {
    const OharaMoeLayer& L = c.layers[l];
    if (L.ff < 0 || (!L.router && L.ff < 1)) return false;
    if (!L.router) {
      act = std::max(act, R * L.ff);
      continue;
    }
    if (L.n_experts < 1 || L.n_experts > 1024 || L.k < 1 || L.k > 16 || L.hidden < 1) return false;
    act = std::max(act, R * L.k * L.hidden);
    act_sh = std::max(act_sh, R * L.ff);
    pairs = std::max(pairs, R * L.k);
    experts = std::max(experts, (int64_t)L.n_experts);
  }
  const bool i8 = c.kvstats != nullptr, wide = c.head_dim == 64 || c.head_dim == 128;
  s.dequantise = i8 && c.seq_len >= 16 && wide;
  s.attend_rows = i8 ? s.dequantise : ohara_attn_prefill_wins(c.batch, c.seq_len, c.n_heads, c.n_kv_heads, c.head_dim, c.pos);
  s.room_bytes = s.attend_rows ? std::max<int64_t>(0, ohara_attn_prefill_ws_bytes(c.batch, c.seq_len, c.n_heads, c.n_kv_heads, c.head_dim, c.pos)) : 0;
  const int64_t heads = (int64_t)c.n_heads * c.head_dim, kv = i8 ? (int64_t)c.n_kv_heads * c.head_dim : 0;
  const uintptr_t at = (uintptr_t)c.scratch;
  s.bytes = 0;
  auto take = [&](auto*& p, int64_t n) {
    p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(at + s.bytes);
    s.bytes += (n * (int64_t)sizeof(*p) + 255) & ~(int64_t)255;
  };
  take(s.x, R * d);
  take(s.y, R * d);
  take(s.xn, R * d);
  take(s.q, R * heads);
  take(s.attn, R * heads);
  take(s.k, R * kv);
  take(s.v, R * kv);
  take(s.kd, s.dequantise ? (int64_t)c.batch * (c.pos + c.seq_len) * kv : 0);
  take(s.vd, s.dequantise ? (int64_t)c.batch * (c.pos + c.seq_len) * kv : 0);
  take(s.w, pairs);
  take(s.act, act);
  take(s.act_sh, act_sh);
  take(s.out, (pairs + R) * d);
  take(s.router, R * experts);
  take(s.idx, pairs);
  take(s.meta, experts + 1 + 2 * pairs);
  unsigned char* room;
  take(room, s.room_bytes);
  s.room = room;
  return true;
}

}  // namespace

extern "C" int64_t ohara_moe_forward_bytes(const OharaMoeCall* c) {
  MoeScratch s;
  return c && moe_scratch(*c, s) ? s.bytes : OHARA_EINVAL;
}

extern "C" int ohara_moe_forward(const OharaMoeCall* cp, void* stream) {
  MoeScratch s;
  if (!cp || !moe_scratch(*cp, s)) return OHARA_EINVAL;
  const OharaMoeCall& c = *cp;
  if (!c.token_emb || !c.final_norm || !c.w_vocab || !c.cos || !c.sin || !c.ids || !c.kcache || !c.vcache || !c.logits) return OHARA_EINVAL;
  if (!c.scratch || ((uintptr_t)c.scratch & 255) || c.scratch_bytes < s.bytes) return OHARA_EINVAL;
  const int B = c.batch, S = c.seq_len, R = B * S, d = c.d_model, H = c.n_heads, Hkv = c.n_kv_heads, Dh = c.head_dim;
  const int n_split = S == 1 ? c.n_split : 1;
  auto ahead = [&](int n) { return ohara_norm_ahead(R, d, (n + 15) / 16 * 16); };
  const bool qkv_normed = ahead((H + 2 * Hkv) * Dh);
  uint16_t *x = s.x, *next = s.y;
  int rc = ohara_embed_bf16(c.ids, c.token_emb, x, R, d, c.vocab, stream);
  for (int l = 0; l < c.n_layers && !rc; ++l) {
    const OharaMoeLayer& L = c.layers[l];
    const uint16_t* rows = qkv_normed ? s.xn : x;
    const uint16_t* norm = qkv_normed ? nullptr : L.norm1;
    if (qkv_normed) rc = ohara_rmsnorm_bf16(x, L.norm1, s.xn, R, d, c.eps, stream);
    if (rc) return rc;
    if (c.kvstats) {
      int8_t *kq = (int8_t*)c.kcache[l], *vq = (int8_t*)c.vcache[l];
      float* stats = (float*)c.kvstats[l];
      rc = ohara_qkv_rope_bf16(rows, d, L.wqkv, d, norm, c.eps, B, S, H, Hkv, Dh, c.cos, c.sin, c.pos, nullptr, c.t_max, s.q, s.k, s.v, stream);
      if (!rc && S > 1) rc = ohara_kv_quant_append_int8(s.k, s.v, B, S, Hkv, Dh, c.pos, nullptr, kq, vq, stats, c.t_max, stream);
      if (S == 1) {
        if (!rc) rc = ohara_attn_append_int8(s.q, s.k, s.v, kq, vq, stats, B, H, Hkv, Dh, c.t_max, c.pos, nullptr, 0, n_split, c.attn_ws, s.attn, stream);
      } else if (s.dequantise) {
        const int len = c.pos + S;
        if (!rc) rc = ohara_kv_dequant_int8(kq, stats, 0, B, len, Hkv, Dh, c.t_max, s.kd, stream);
        if (!rc) rc = ohara_kv_dequant_int8(vq, stats, 1, B, len, Hkv, Dh, c.t_max, s.vd, stream);
        if (!rc) rc = ohara_attn_prefill_ws_bf16(s.q, s.kd, s.vd, B, S, H, Hkv, Dh, len, c.pos, s.attn, s.room, s.room_bytes, stream);
      } else if (!rc) {
        rc = ohara_attn_cached_int8(s.q, kq, vq, stats, B, S, H, Hkv, Dh, c.t_max, c.pos, nullptr, n_split, c.attn_ws, s.attn, stream);
      }
    } else {
      uint16_t *kc = (uint16_t*)c.kcache[l], *vc = (uint16_t*)c.vcache[l];
      rc = ohara_qkv_rope_append_bf16(rows, d, L.wqkv, d, norm, c.eps, B, S, H, Hkv, Dh, c.cos, c.sin, c.pos, nullptr, s.q, kc, vc, c.t_max, stream);
      if (!rc && s.attend_rows)
        rc = ohara_attn_prefill_ws_bf16(s.q, kc, vc, B, S, H, Hkv, Dh, c.t_max, c.pos, s.attn, s.room, s.room_bytes, stream);
      else if (!rc)
        rc = ohara_attn_cached_bf16(s.q, kc, vc, B, S, H, Hkv, Dh, c.t_max, c.pos, nullptr, n_split, c.attn_ws, s.attn, stream);
    }
    if (!rc) rc = ohara_gemm_skinny_bf16(s.attn, H * Dh, L.wo, d, H * Dh, nullptr, c.eps, R, OHARA_EPI_RESIDUAL, x, d, x, d, stream);
    if (rc) return rc;
    if (!L.router) {
      const bool gu_normed = ahead(2 * ((L.ff + 7) / 8 * 8));
      if (gu_normed) rc = ohara_rmsnorm_bf16(x, L.norm2, s.xn, R, d, c.eps, stream);
      if (!rc) rc = ohara_gemm_skinny_bf16(gu_normed ? s.xn : x, d, L.wgu, L.ff, d, gu_normed ? nullptr : L.norm2, c.eps, R, OHARA_EPI_SWIGLU, nullptr, 0, s.act, L.ff, stream);
      if (!rc) rc = ohara_gemm_skinny_bf16(s.act, L.ff, L.wdown, d, L.ff, nullptr, c.eps, R, OHARA_EPI_RESIDUAL, x, d, x, d, stream);
      continue;
    }
    const int pairs = R * L.k, E = L.n_experts;
    int32_t *offs = s.meta, *pair_of = offs + E + 1, *pos_of = pair_of + pairs;
    uint16_t* y_sh = L.wgu ? s.out + (size_t)pairs * d : nullptr;
    if (E <= 64 && pairs <= 1024 && d <= 4096 && !((d | L.hidden | L.ff) & 7)) {
      rc = ohara_moe_route_fused(x, d, L.norm2, c.eps, L.router, L.router_bias, R, d, E, L.k, L.biased_topk, L.gate_sigmoid, L.normalize, s.xn, d,
                                 nullptr, E, s.idx, s.w, offs, pair_of, pos_of, L.counter, stream);
      if (!rc) rc = ohara_moe_experts_gate_up_shared(s.xn, d, L.experts_gu, L.gu_stride, E, L.hidden, d, L.k, offs, pair_of, s.act, L.hidden, L.wgu,
                                                     L.wgu ? L.ff : 0, R, L.wgu ? s.act_sh : nullptr, L.ff, stream);
      if (!rc) rc = ohara_moe_experts_down_shared(s.act, L.hidden, L.experts_down, L.down_stride, E, d, L.hidden, L.k, offs, pair_of, s.w, s.out, d,
                                                  L.wgu ? L.wdown : nullptr, L.wgu ? L.ff : 0, R, L.wgu ? s.act_sh : nullptr, L.ff, y_sh, d, stream);
    } else {
      rc = ohara_rmsnorm_bf16(x, L.norm2, s.xn, R, d, c.eps, stream);
      if (!rc) rc = ohara_gemm_skinny_bf16(s.xn, d, L.router, E, d, nullptr, c.eps, R, OHARA_EPI_STORE, nullptr, 0, s.router, E, stream);
      if (!rc) rc = ohara_moe_route_topk(s.router, E, L.router_bias, R, E, L.k, L.biased_topk, L.gate_sigmoid, L.normalize, s.idx, s.w, stream);
      if (!rc) rc = ohara_moe_sort_pairs(s.idx, pairs, E, offs, pair_of, pos_of, stream);
      if (!rc) rc = ohara_moe_experts_gate_up_many(s.xn, d, L.experts_gu, L.gu_stride, E, L.hidden, d, L.k, pairs, offs, pair_of, s.act, L.hidden, stream);
      if (!rc) rc = ohara_moe_experts_down_many(s.act, L.hidden, L.experts_down, L.down_stride, E, d, L.hidden, L.k, pairs, offs, pair_of, s.w, s.out, d,
                                                stream);
      if (!rc && L.wgu) rc = ohara_gemm_skinny_bf16(s.xn, d, L.wgu, L.ff, d, nullptr, c.eps, R, OHARA_EPI_SWIGLU, nullptr, 0, s.act_sh, L.ff, stream);
      if (!rc && L.wgu) rc = ohara_gemm_skinny_bf16(s.act_sh, L.ff, L.wdown, d, L.ff, nullptr, c.eps, R, OHARA_EPI_STORE, nullptr, 0, y_sh, d, stream);
    }
    if (!rc) rc = ohara_moe_combine(s.out, d, s.idx, pos_of, R, L.k, y_sh, d, x, d, next, d, d, stream);
    std::swap(x, next);
  }
  if (rc) return rc;
  // the last token of every sequence: a strided view, normed by the projection
  const bool last = c.last_only && S > 1;
  const bool normed = !last && ahead(c.vocab);
  if (normed) rc = ohara_rmsnorm_bf16(x, c.final_norm, s.xn, R, d, c.eps, stream);
  if (rc) return rc;
  return ohara_gemm_skinny_bf16(normed ? s.xn : last ? x + (size_t)(S - 1) * d : x, last ? S * d : d, c.w_vocab, c.vocab, d,
                                normed ? nullptr : c.final_norm, c.eps, last ? B : R, OHARA_EPI_STORE, nullptr, 0, c.logits, c.vocab, stream);
}
