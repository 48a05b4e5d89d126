/*
 * ohara_decode.h - C ABI of libohara_decode.so, the MI355X (gfx950) kernels behind
 * ohara's KV-cache decode path.
 *
 * The reference (joey00072/ohara) is pure Python/PyTorch and has no FFI of its own;
 * each entry point below names the reference code it replaces (file:line in the
 * reference tree).  Conventions shared by every function:
 *
 *   - plain C: raw device pointers, sizes, a hipStream_t passed as void*;
 *   - returns OHARA_OK (0) or a negative OHARA_E* code; never throws, never exits,
 *     never allocates or frees device memory, and does not synchronise the host (the one
 *     exception is the one-time workspace set-up ohara_llama_decode_persistent(init_workspace=1));
 *   - all work is enqueued on `stream` and is stream-ordered, so every call can be
 *     recorded into a HIP graph;
 *   - bf16 tensors are passed as uint16_t* (raw bfloat16 bits), row-major;
 *   - `pos_dev` arguments: when non-NULL the kernel reads the cache position of the
 *     token being fed from that device int32 instead of the host argument (the
 *     visible length is then *pos_dev + 1), so a captured graph can be replayed
 *     while the position advances on the device.
 *
 * Weight matrices of Linear layers are consumed in a packed tile order produced by
 * ohara_pack_rows_bf16 (see below); everything else is in the reference's layout.
 */
#ifndef OHARA_DECODE_H
#define OHARA_DECODE_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define OHARA_OK 0
#define OHARA_EINVAL (-1)   /* an argument violates the documented constraints */
#define OHARA_ELAUNCH (-2)  /* the HIP runtime rejected a launch */
#define OHARA_ESIZE (-3)    /* a size exceeds what the entry point supports */

/* Library version and a self-description string (build flags, arch). */
int ohara_abi_version(void);

/* ---- weight packing -------------------------------------------------------
 * Packed layout "strip/kstep/lane": the (N, K) row-major bf16 matrix of a Linear
 * (nn.Linear.weight, ohara/models/llama.py:60-63,252; ohara/modules/mlp.py:146-148)
 * is cut into strips of 16 rows and k-steps of 32 columns; the tile (strip s,
 * k-step j) is stored as 64 lanes x 8 bf16, lane = 16*g + m holding row
 * perm[16*s + m], columns 32*j + 8*g .. +7.  N is padded to a multiple of 16 and
 * K to a multiple of 32 with zeros.  `perm` (length padded N, int32, source row or
 * -1 for a zero row) may be NULL for the identity.
 * Returns the packed size in bytes through *bytes when `dst` is NULL. */
int ohara_pack_rows_bf16(const uint16_t* w, int n, int k, int ldw, const int32_t* perm, int n_padded,
                         uint16_t* dst, int64_t* bytes, void* stream);

/* ---- embedding ------------------------------------------------------------
 * out[t, :] = table[ids[t], :]            (nn.Embedding, llama.py:245,310) */
int ohara_embed_bf16(const int64_t* ids, const uint16_t* table, uint16_t* out, int n_tokens, int d, int vocab,
                     void* stream);

/* ---- RMSNorm --------------------------------------------------------------
 * out = bf16(x * rsqrt(mean(x^2) + eps)) * w      (ohara/modules/norm.py:16-21) */
int ohara_rmsnorm_bf16(const uint16_t* x, const uint16_t* w, uint16_t* out, int rows, int d, float eps,
                       void* stream);

/* ---- skinny GEMM (decode projections) ------------------------------------------
 * y = [rmsnorm(x; norm_w, eps)] @ W^T  with one of three epilogues.  `wp` is W in
 * the packed layout; n / k are the logical sizes of W.  norm_w may be NULL.
 * `batch` rows of x.  More than 64 rows without a fused norm (without a residual and with
 * k > 1024: more than 16) go to the tiled MFMA kernel of ohara_gemm_bf16; with a fused norm they are processed 64 at a time, each
 * chunk streaming W once.
 *
 * OHARA_EPI_STORE      out[b, n] = bf16(y)                      (any Linear)
 * OHARA_EPI_RESIDUAL   out[b, n] = bf16(resid[b, n] + bf16(y))  (llama.py:199-200)
 * OHARA_EPI_SWIGLU     W packed with gate/up rows interleaved (ohara_swiglu_perm);
 *                      out[b, f] = bf16(bf16(silu(bf16(gate))) * bf16(up))
 *                                                               (mlp.py:152)
 * The fused QKV + rotary + cache append is a separate entry point below. */
#define OHARA_EPI_STORE 0
#define OHARA_EPI_RESIDUAL 1
#define OHARA_EPI_SWIGLU 2
int ohara_gemm_skinny_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* norm_w,
                           float eps, int batch, int epilogue, const uint16_t* resid, int ldr, uint16_t* out,
                           int ldo, void* stream);

/* Row permutation that interleaves gate and up rows for OHARA_EPI_SWIGLU: packed
 * row 16*s + 4*g + i is gate row 8*s + 2*g + i (i < 2) or up row 8*s + 2*g + i - 2.
 * Source rows index the vertical concatenation [gate; up] of two (f, k) matrices.
 * perm has 2 * f_padded entries, f_padded = f rounded up to a multiple of 8. */
int ohara_swiglu_perm(int f, int32_t* perm_host);

/* ---- tiled MFMA GEMM (batched prefill projections) ---------------------------
 * out = epi(x @ W^T) for any number of rows: output tiles of 32 x 32 to 256 x 256, the one that a model of the times
 * says is fastest, K in steps of 64 or 128, activations and packed weights both straight into LDS.
 * Same packed `wp`, same epilogues and the same rounding points as ohara_gemm_skinny_bf16
 * (llama.py:84-86,142,322, mlp.py:152 with more than one position per call).  No fused norm. */
int ohara_gemm_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, int rows, int epilogue,
                    const uint16_t* resid, int ldr, uint16_t* out, int ldo, void* stream);
/* 1 where rows are best normed ahead of their projection (norm_w then NULL) and not by it: more than 64, more than 32 where k > 1024 and the
 * packed rows are many, more than 16 where k > 2048.  What ohara_llama_forward does by itself. */
int ohara_projection_norm_ahead(int rows, int k, int packed_rows);
/* The tile of such a product over rows that start on 16 bytes: 1000 * its rows + its packed rows (SwiGLU packs two a column).  Under 1024 rows and from 20000
 * packed rows on the call below says which one a plain store runs. */
int ohara_gemm_tile_of(int rows, int packed_rows, int k);
/* The same of a product with an epilogue (as below), or of its sums in parts of the depth (parts > 1, which divide k; then the epilogue does not matter);
 * 1 more where it is one of the tiles in halves. */
int ohara_gemm_tile_with(int rows, int packed_rows, int k, int epilogue, int parts);
/* How many of the rows go first, where they take two launches (0: one).  epilogue: 0 store, 1 residual, 2 SwiGLU, 3 rotary with heads of dh, 4 bias, 6 bias and
 * two addends, 5 and 7 to 11 the arithmetic ones (bias and gelu, Phi's input, soft cap, gelu times an embedding, gated units, two-sided activation). */
int ohara_gemm_first_rows(int rows, int packed_rows, int k, int epilogue, int dh);

/* Fused q/k/v projection + rotary + KV-cache append: replaces Attention.forward's
 * three Linears, apply_rope and KVCache.forward (llama.py:84-98;
 * ohara/embeddings_pos/rotary.py:55-93; ohara/modules/kv_cache.py:75-118).
 * x holds batch*seq_len rows, row b*seq_len + s being position pos + s of sequence b
 * (seq_len = 1 at decode).  `wp` packs the rows [W_q; W_k; W_v].
 *   q_out  (batch*seq_len, h*dh) bf16, rotated
 *   kcache/vcache (batch_cap, t_max, h_kv, dh) bf16; rows pos..pos+seq_len-1 of
 *   sequence b are written with the rotated keys / the values.
 * cos/sin: (>= pos+seq_len, dh/2) bf16 tables (precompute_freqs_cis, rotary.py:24-38). */
int ohara_qkv_rope_append_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w,
                               float eps, int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                               const uint16_t* sin, int pos, const int32_t* pos_dev, uint16_t* q_out,
                               uint16_t* kcache, uint16_t* vcache, int t_max, void* stream);

/* The same projection + rotary, with the rotated k and the v rows written to (batch*seq_len,
 * h_kv*dh) buffers instead of into a cache (the int8 cache quantises them in a second step).
 * t_max only bounds the positions. */
/* ohara_qkv_rope_append_bf16 with one cache position per sequence: token s of sequence b is
 * rotated for, and appended at, position seq_pos[b] + s (device array, `batch` entries). */
int ohara_qkv_rope_append_ragged_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w,
                                      float eps, int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                                      const uint16_t* sin, const int32_t* seq_pos, uint16_t* q_out, uint16_t* kcache,
                                      uint16_t* vcache, int t_max, void* stream);
/* Rows of prompts side by side (always the tiled kernel, no norm): `at` (device) holds the position of every row, then the
 * row of the caches that its sequence is in. */
int ohara_qkv_rope_append_rows_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, int rows, int h, int h_kv, int dh,
                                    const uint16_t* cos, const uint16_t* sin, const int32_t* at, uint16_t* q_out, uint16_t* kcache,
                                    uint16_t* vcache, int t_max, void* stream);
int ohara_qkv_rope_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w, float eps,
                        int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos, const uint16_t* sin,
                        int pos, const int32_t* pos_dev, int t_max, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out,
                        void* stream);

/* ohara_qkv_rope_bf16 with one position per sequence (seq_pos as in ohara_qkv_rope_append_ragged_bf16). */
int ohara_qkv_rope_ragged_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w, float eps,
                               int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos, const uint16_t* sin,
                               const int32_t* seq_pos, int t_max, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out,
                               void* stream);

/* ---- attention over the KV cache ------------------------------------------------
 * Query s (0 <= s < seq_len) of sequence b sits at cache position pos + s and sees
 * positions [0, pos + s] (the cache mask key_pos <= start_pos + q_idx, llama.py:109-113):
 *   out[b, s, h, :] = softmax(q[b,s,h,:] . K[b, 0:pos+s+1, h/(H/Hkv), :] / sqrt(dh)) V
 * (llama.py:100-135; GQA by head indexing instead of repeat_interleave :101-103).
 * seq_len = 1 is the decode case.  The context is split into at most `n_split` chunks
 * (dh 64 and 128: as many as its length at the call asks for; otherwise `n_split`);
 * partial (max, sum, acc) triples go to `workspace` and the last chunk to finish
 * merges them in chunk order.  workspace bytes = ohara_attn_workspace_bytes(
 * batch*seq_len, h, h_kv, dh, n_split); zero-fill it once before first use (the
 * kernels leave its counters at zero).  n_split = 1 needs no workspace (NULL ok);
 * n_split > 1 needs (h / h_kv) * n_split <= 2048.
 * q / out: (batch*seq_len, h*dh). */
int64_t ohara_attn_workspace_bytes(int batch, int h, int h_kv, int dh, int n_split);
int ohara_attn_cached_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch,
                           int seq_len, int h, int h_kv, int dh, int t_max, int pos, const int32_t* pos_dev,
                           int n_split, void* workspace, uint16_t* out, void* stream);
/* The same with one position per sequence: query s of sequence b sits at seq_pos[b] + s and sees
 * [0, seq_pos[b] + s].  No counterpart in the reference (one scalar position, llama.py:287-299). */
int ohara_attn_cached_ragged_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch,
                                  int seq_len, int h, int h_kv, int dh, int t_max, const int32_t* seq_pos, int n_split,
                                  void* workspace, uint16_t* out, void* stream);
/* seq_pos[b] += by for every b with active[b] != 0 (active NULL: all): advances a ragged batch by one
 * decode step without host involvement (graph replay). */
int ohara_advance_positions(int32_t* seq_pos, const uint8_t* active, int batch, int by, void* stream);
/* The same in one launch with the next step's inputs: next_ids[b] = new_ids[b] for an active sequence, 0 for
 * an idle slot (it rides along at position 0).  No counterpart in the reference (one position for the batch). */
int ohara_advance_ragged(int32_t* seq_pos, const uint8_t* active, const int64_t* new_ids, int64_t* next_ids, int batch,
                         int by, void* stream);
/* Slots of a ragged batch that are taken or left, in one launch: seq_pos[slots[i]] = positions[i] (NULL: 0), active_flags[slots[i]] = active,
 * next_ids[slots[i]] = ids[i] (NULL: as it is if active, else 0).  slots and positions lie on the host and may change when the call returns;
 * ids, next_ids, seq_pos and active_flags on the device.  No counterpart in the reference (one position for the batch). */
int ohara_set_slots(const int32_t* slots, const int32_t* positions, int n, int active, const int64_t* ids, int64_t* next_ids,
                    int32_t* seq_pos, uint8_t* active_flags, int batch, void* stream);

/* ohara_attn_cached_bf16 for callers that cannot allocate device memory (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc).  It has no counterpart in the
 * reference.  Same arguments minus the workspace: the chunk partials and counters live in a
 * device array inside the library (8 MiB + 64 KiB, held by every GPU the library runs on until
 * the process ends), so nothing is allocated or freed, by this library or through any other.
 * Limits: batch*seq_len*h_kv <= 16384 and
 *   align256(batch*seq_len*h*n_split*8) + align256(batch*seq_len*h*n_split*dh*4) <= 8 MiB;
 * anything larger returns OHARA_ESIZE and launches nothing.  The first call on a device looks up
 * the array's address (make it outside graph capture).  All calls on one GPU share the array:
 * calls that overlap in time on one GPU (different streams) race; calls on one stream do not. */
int ohara_attn_cached_bf16_noalloc(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch,
                                   int seq_len, int h, int h_kv, int dh, int t_max, int pos, const int32_t* pos_dev,
                                   int n_split, uint16_t* out, void* stream);

/* Same contract for many query positions per sequence (prefill), as a causal flash-style kernel
 * on MFMA: 16 to 128 queries per workgroup, keys/values walked in 64-position tiles through LDS,
 * online softmax in fp32, probabilities rounded to bf16 for the second product.  dh 64 or 128.
 * Needs no workspace.  (llama.py:100-135 with S > 1.) */
int ohara_attn_prefill_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch,
                            int seq_len, int h, int h_kv, int dh, int t_max, int pos, uint16_t* out, void* stream);
/* The same with room for partial results (16-byte aligned; ohara_attn_prefill_ws_bytes of `pos` or a later one, 0: none needed): few
 * queries behind a long context are then cut into chunks of positions over more workgroups.  Too little room or NULL: as without. */
int64_t ohara_attn_prefill_ws_bytes(int batch, int seq_len, int h, int h_kv, int dh, int pos);
int ohara_attn_prefill_ws_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int batch, int seq_len, int h,
                               int h_kv, int dh, int t_max, int pos, uint16_t* out, void* workspace, int64_t workspace_bytes, void* stream);
/* 1 where they are the faster ones of the two (and take the sizes): ohara_attn_cached_bf16 reads the context once for every token.
 * _with: for a call that has this much room; the other one for one that has what it asks for. */
int ohara_attn_prefill_wins(int batch, int seq_len, int h, int h_kv, int dh, int pos);
int ohara_attn_prefill_wins_with(int batch, int seq_len, int h, int h_kv, int dh, int pos, int64_t workspace_bytes);

/* ohara_attn_prefill_bf16 over n prompts of their own lengths, their query rows side by side, each from position 0 of its row of the
 * caches: `lengths` on the host; `seqs` on the device: n first query rows, n lengths, n rows of the caches. */
int ohara_attn_prompts_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int n, const int32_t* lengths,
                            const int32_t* seqs, int h, int h_kv, int dh, int t_max, uint16_t* out, void* stream);


/* ---- int8 KV cache (ohara/modules/kv_cache.py:15-32, 67-73, 94-102, 116-118) ------------------
 * Every (sequence, position, head) row of dh values is stored as int8 with an fp32 scale and
 * minimum: scale = max((max - min) / 255, 1e-8), q = clamp(round((x - min) / scale - 128), -128,
 * 127), read back as bf16((q + 128) * scale + min).  The quantisation arithmetic is rounded to
 * bf16 after every operation, as the reference's tensor ops on a bf16 cache are, so codes, scales
 * and minima are bit-identical to it.  Caches: (batch_cap, t_max, h_kv, dh) int8.  Statistics:
 * `stats`, (batch_cap, h_kv, t_max, 4) fp32 = one 16-byte record (key scale, key minimum, value
 * scale, value minimum) per row, consecutive positions of a head contiguous (the order decode
 * attention reads them in; the reference's four (B, T, H_kv, 1) tensors, kv_cache.py:67-73, are
 * strided views of it).
 *   ohara_kv_quant_append_int8  quantises k / v rows (batch*seq_len, h_kv*dh) into positions
 *                               pos + s (pos_dev as elsewhere);
 *   ohara_kv_dequant_int8       the first `len` positions of the key (which = 0) or value (which = 1)
 *                               cache tensor as bf16 (batch, len, h_kv, dh) - what KVCache._read returns;
 *   ohara_attn_cached_int8      ohara_attn_cached_bf16 over the quantised cache, dequantising in
 *                               registers.  Scales must be bf16-representable, as the quantiser
 *                               writes them: (q + 128) * scale is then exact in fp32 and the
 *                               kernel's fused multiply-add equals the reference's two roundings. */
int ohara_kv_quant_append_int8(const uint16_t* k, const uint16_t* v, int batch, int seq_len, int h_kv, int dh, int pos,
                               const int32_t* pos_dev, int8_t* kq, int8_t* vq, float* stats, int t_max, void* stream);
int ohara_kv_dequant_int8(const int8_t* q, const float* stats, int which, int batch, int len, int h_kv, int dh,
                          int t_max, uint16_t* out, void* stream);
int ohara_attn_cached_int8(const uint16_t* q, const int8_t* kcache, const int8_t* vcache, const float* stats, int batch,
                           int seq_len, int h, int h_kv, int dh, int t_max, int pos, const int32_t* pos_dev, int n_split,
                           void* workspace, uint16_t* out, void* stream);
/* ohara_kv_quant_append_int8 of one position a sequence (pos_stride 1: ohara_kv_quant_append_ragged_int8's, pos_dev the positions) and the
 * attention of its queries, in one launch where heads are 64 or 128 wide, in groups of 1, 2 or 4. */
int ohara_attn_append_int8(const uint16_t* q, const uint16_t* k, const uint16_t* v, int8_t* kcache, int8_t* vcache, float* stats, int batch,
                           int h, int h_kv, int dh, int t_max, int pos, const int32_t* pos_dev, int pos_stride, int n_split, void* workspace,
                           uint16_t* out, void* stream);

/* The append and the attention with one cache position per sequence (seq_pos: device array, `batch`
 * entries; token s of sequence b goes to / sits at seq_pos[b] + s).  No counterpart in the reference,
 * whose forward takes one scalar position for the whole batch (llama.py:287-299); the cache itself
 * (kv_cache.py:94-118) is indifferent to where each sequence stands. */
int ohara_kv_quant_append_ragged_int8(const uint16_t* k, const uint16_t* v, int batch, int seq_len, int h_kv, int dh,
                                      const int32_t* seq_pos, int8_t* kq, int8_t* vq, float* stats, int t_max,
                                      void* stream);
int ohara_attn_cached_ragged_int8(const uint16_t* q, const int8_t* kcache, const int8_t* vcache, const float* stats,
                                  int batch, int seq_len, int h, int h_kv, int dh, int t_max, const int32_t* seq_pos,
                                  int n_split, void* workspace, uint16_t* out, void* stream);

/* ---- greedy selection ---------------------------------------------------------
 * next_ids[b] = first index of max(logits[b, 0:valid_vocab])  (argmax of the last
 * position, ohara/chat_engine.py:61-63, ohara/inference.py:40-45; ids >= valid_vocab
 * are the padded vocabulary masked at chat_engine.py:398-399).  When `step_state`
 * (device, 4 x int32: pos, step, done, pad) is given, the token is also written to
 * history[step * batch + b] (if step < hist_cap) and the last workgroup to finish
 * advances pos and step by one - the device-side loop bookkeeping. */
int ohara_argmax_bf16(const uint16_t* logits, int ldl, int batch, int vocab, int valid_vocab, int64_t* next_ids,
                      int64_t* history, int hist_cap, int32_t* step_state, void* stream);

/* ---- temperature / top-k / top-p sampling ------------------------------------------
 * sample_next_token (ohara/chat_engine.py:51-82) and the nucleus branch of
 * Inference.sampler (ohara/inference.py:46-64) for temperature > 0, fused into one
 * launch, one workgroup per row:
 *   x = logits / temperature, ids >= valid_vocab masked (:398-399); top_k > 0 keeps
 *   x >= the k-th largest (ties survive, :66-69); p = softmax(x); 0 < top_p < 1 keeps the
 *   smallest descending-sorted prefix whose preceding mass does not exceed top_p
 *   (:72-81), renormalised; otherwise all of p in vocabulary order (:82).
 * torch.multinomial is replaced by inverse-CDF sampling with the caller's uniform draw
 * u[b] in [0,1); equal probabilities are ordered lowest id first.  Deterministic.
 * logits: (batch, vocab) bf16 (logits_are_fp32 = 0) or fp32.  vocab <= 131072.
 * history / step_state as in ohara_argmax_bf16.  With step_state and u_step_stride > 0 the draw of
 * row b is u[step * u_step_stride + b] (step = index of the token being produced, read on the
 * device), so a captured decode loop walks a pre-drawn (steps, batch) tensor by itself;
 * otherwise u[b].  temperature == 0 is ohara_argmax_bf16. */
int ohara_sample_topk_topp(const void* logits, int logits_are_fp32, int ldl, int batch, int vocab,
                           int valid_vocab, float temperature, int top_k, float top_p, const float* u,
                           int u_step_stride, int64_t* out_ids, int64_t* history, int hist_cap,
                           int32_t* step_state, void* stream);
/* The same selection, same results, for a caller whose sampler calls on one GPU do not overlap in time
 * (one decode stream, as in ohara/chat_engine.py's generate loop): a small top-k (<= 64) on a long bf16
 * row (8192 < vocab <= 65536, batch <= 64) is spread over one workgroup per 8192 ids, whose candidates
 * meet in a 330 KB scratch array inside the library (nothing is allocated); every other shape runs
 * ohara_sample_topk_topp's kernels.  Overlapping calls of this entry point on one GPU would share
 * that array. */
int ohara_sample_topk_topp_exclusive(const void* logits, int logits_are_fp32, int ldl, int batch, int vocab,
                           int valid_vocab, float temperature, int top_k, float top_p, const float* u,
                           int u_step_stride, int64_t* out_ids, int64_t* history, int hist_cap,
                           int32_t* step_state, void* stream);
/* The same spread selection with the candidates meeting in the CALLER's workspace instead of the library's
 * array: calls with different workspaces may overlap in time (one workspace per decode session / stream).
 * workspace: ohara_sample_workspace_bytes() bytes of device memory, 256-byte aligned, zeroed once before its
 * first use (the kernels leave its counters at zero); calls sharing one workspace must not overlap. */
int64_t ohara_sample_workspace_bytes(void);
int ohara_sample_topk_topp_ws(const void* logits, int logits_are_fp32, int ldl, int batch, int vocab,
                              int valid_vocab, float temperature, int top_k, float top_p, const float* u,
                              int u_step_stride, int64_t* out_ids, int64_t* history, int hist_cap,
                              int32_t* step_state, void* workspace, int64_t workspace_bytes, void* stream);

/* ---- BitNet-b1.58 BitLinear (ternary weights x int8 activations, int32 accumulate) ------
 * Integer form of BitLinear.forward (experiments/bitnet/bitnet.py:29-59):
 *   x_hat = RMSNorm(x; norm_w, eps) in bf16 (:49,53); s = 127 / max(max|x_hat|, 1e-5) and
 *   q = clamp(rint(x_hat * s), -128, 127) per row (:30-33); acc[n] = sum_k q[k] * T[n,k] in
 *   int32; y = bf16((float(acc) / s) * gamma) [+ resid]  (:58-59, bias dropped).
 * T in {-1,0,1} and gamma = max(mean|W|, 1e-5) come from weight_quant (:37-43), done once at
 * load time.  ohara_bitlinear_pack_ternary turns T (n, k) int8 row-major into the packed
 * 2-bit stream the kernels read (16 weights per dword; size through *bytes when dst is NULL).
 * ohara_act_quant_int8 and ohara_gemv_ternary_i8 are the two halves; ohara_bitlinear_bf16
 * fuses them (k <= 6144).  acc_out, when given, receives the raw int32 accumulators - the
 * quantity that must match a CPU int32 matmul bit for bit.  ldq must be a multiple of 16,
 * k and ldx multiples of 8.  pre_norm_w (may be NULL) is the weight of the block-level RMSNorm
 * that precedes the projection (llama.py:199-200), applied in the same pass: x := bf16(
 * RMSNorm(x; pre_norm_w, eps)) before the BitLinear's own norm. */
int ohara_bitlinear_pack_ternary(const int8_t* t, int n, int k, int ldt, uint32_t* dst, int64_t* bytes, void* stream);
int ohara_act_quant_int8(const uint16_t* x, int ldx, const uint16_t* norm_w, float eps, int rows, int k, int8_t* q,
                         int ldq, float* s, int32_t* sumq, void* stream);
int ohara_gemv_ternary_i8(const int8_t* q, int ldq, const float* s, const int32_t* sumq, const uint32_t* wp, int n,
                          int k, float gamma, int rows, const uint16_t* resid, int ldr, uint16_t* out, int ldo,
                          int32_t* acc_out, int ldacc, void* stream);
/* Many rows: each row quantised once for each of `sets` (at most three) BitLinears that read it and differ in their norm
 * weight; q: (sets, rows, ldq), s and sumq: (sets, rows).  ohara_gemv_ternary_i8 (more than 12 rows, q on 16 bytes),
 * ohara_gemm_ternary_sets_i8 (`sets` weights of n columns, one output each) and ohara_gemm_ternary_qkv_rope_append (query, key,
 * value: rotary + append as in ohara_bitlinear_qkv_rope_append_bf16, any number of rows) multiply the codes in tiles; the
 * accumulators are those of ohara_bitlinear_bf16.  ldq a multiple of 16, q on 16 bytes, k a multiple of 8. */
int ohara_act_quant_sets_int8(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, const uint16_t* const* norm_w, int sets,
                              float eps, int rows, int k, int8_t* q, int ldq, float* s, int32_t* sumq, void* stream);
/* The same for one BitLinear whose input rows are bf16(bf16(silu(gate)) * up) (ohara/modules/mlp.py:152); gate and up: rows ld apart. */
int ohara_act_quant_swiglu_int8(const uint16_t* gate, const uint16_t* up, int ld, const uint16_t* norm_w, float eps, int rows, int k,
                                int8_t* q, int ldq, float* s, int32_t* sumq, void* stream);
int ohara_gemm_ternary_sets_i8(const int8_t* q, int ldq, const float* s, const int32_t* sumq, const uint32_t* const* wp,
                               const float* gamma, int sets, int n, int k, int rows, uint16_t* const* out, int ldo, void* stream);
int ohara_gemm_ternary_qkv_rope_append(const int8_t* q, int ldq, const float* s, const int32_t* sumq, const uint32_t* const* wp,
                                       const float* gamma, int k, int batch, int seq_len, int h, int h_kv, int dh,
                                       const uint16_t* cos, const uint16_t* sin, int pos, const int32_t* pos_dev, uint16_t* q_out,
                                       uint16_t* kcache, uint16_t* vcache, int t_max, void* stream);
int ohara_bitlinear_bf16(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, const uint16_t* norm_w, float eps,
                         const uint32_t* wp, int n, int k, float gamma, int rows, const uint16_t* resid, int ldr,
                         uint16_t* out, int ldo, int32_t* acc_out, int ldacc, void* stream);

/* Groups of BitLinears that read the same rows, for decode (rows <= 64), one launch each:
 *   - attn.query / attn.key / attn.value (each with its own norm weight, packed weights and gamma,
 *     index 0..2 of the three arrays) with rotary + cache append as the epilogue: q_out
 *     (rows, h*dh) rotated, rotated k and v written at cache position pos + s (pos_dev as in
 *     ohara_qkv_rope_append_bf16);
 *   - ff.gate and ff.up with SwiGLU as the epilogue: out[b, f] = bf16(bf16(silu(gate)) * up).
 * Same arithmetic as the separate calls (bitnet.py:29-59, rotary.py:55-93, kv_cache.py:104-105,
 * mlp.py:152). */
int ohara_bitlinear_qkv_rope_append_bf16(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, float eps, int k,
                                         const uint16_t* const* norm_w, const uint32_t* const* wp, const float* gamma,
                                         int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                                         const uint16_t* sin, int pos, const int32_t* pos_dev, uint16_t* q_out,
                                         uint16_t* kcache, uint16_t* vcache, int t_max, void* stream);
int ohara_bitlinear_gate_up_bf16(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, float eps, int k, int f,
                                 const uint16_t* gate_norm_w, const uint32_t* gate_wp, float gate_gamma,
                                 const uint16_t* up_norm_w, const uint32_t* up_wp, float up_gamma, int rows,
                                 uint16_t* out, int ldo, void* stream);

/* out = bf16(bf16(silu(gate)) * up), elementwise over n values (ohara/modules/mlp.py:152). */
int ohara_silu_mul_bf16(const uint16_t* gate, const uint16_t* up, uint16_t* out, int64_t n, void* stream);

/* Rotary on q (in place) and on k, and append of the rotated k and of v to the cache, for
 * projections that were computed unfused (ohara/embeddings_pos/rotary.py:55-93,
 * ohara/modules/kv_cache.py:104-105).  q: (batch*seq_len, h*dh), k/v: (batch*seq_len, h_kv*dh).
 * t_max == 0: kcache / vcache are row buffers of k's and v's shape instead of caches - the rotated
 * keys and the values of this call, which an int8 cache's append (ohara_kv_quant_append_int8,
 * kv_cache.py:94-102) takes next; the caller keeps pos + seq_len within the rotary tables. */
int ohara_rope_append_bf16(uint16_t* q, const uint16_t* k, const uint16_t* v, int batch, int seq_len, int h, int h_kv,
                           int dh, const uint16_t* cos, const uint16_t* sin, int pos, const int32_t* pos_dev,
                           uint16_t* kcache, uint16_t* vcache, int t_max, void* stream);

/* ---- grouped mixture-of-experts feed-forward (eval mode) -------------------------------------
 * GroupedMoE.forward (ohara/modules/moe_grouped.py:209-228) in five launches:
 *  ohara_moe_route_topk     _route (:122-147) from the bf16 router logits (n_tokens, n_experts):
 *                           experts = top-k of logits [+ router_bias when biased_topk] with ties
 *                           to the lowest id; weights = softmax (or sigmoid, optionally normalised)
 *                           of the k selected unbiased logits, cast to bf16.  k <= 16, E <= 1024.
 *  ohara_moe_sort_pairs     the stable sort by expert of :161-168: offsets (E+1), pair_of[sorted
 *                           position] = token*k + slot, pos_of = its inverse.  n_pairs <= 65536.
 *  ohara_moe_experts_gate_up  act[sorted position] = bf16(silu(bf16(x W_gate[e]))) * bf16(x W_up[e])
 *  ohara_moe_experts_down     y[sorted position]   = bf16(bf16(act W_down[e]) * weight)   (:175-181)
 *                           expert weights: per expert, rows packed by ohara_pack_rows_bf16
 *                           (gate/up rows interleaved with ohara_swiglu_perm), experts
 *                           expert_stride_bytes apart.
 *  ohara_moe_combine        out[token] = resid + (sum over its experts in ascending expert id,
 *                           each add rounded to bf16 (:184) + shared[token]); shared / resid may
 *                           be NULL. */
int ohara_moe_route_topk(const uint16_t* router_logits, int ldl, const uint16_t* router_bias, int n_tokens, int n_experts,
                         int k, int biased_topk, int gate_sigmoid, int normalize, int32_t* expert_idx,
                         uint16_t* expert_w, void* stream);
int ohara_moe_sort_pairs(const int32_t* expert_idx, int n_pairs, int n_experts, int32_t* offsets, int32_t* pair_of,
                         int32_t* pos_of, void* stream);
int ohara_moe_experts_gate_up(const uint16_t* x, int ldx, const uint16_t* wp_gate_up, int64_t expert_stride_bytes,
                              int n_experts, int hidden, int d, int k, const int32_t* offsets, const int32_t* pair_of,
                              uint16_t* act, int ld_act, void* stream);
int ohara_moe_experts_down(const uint16_t* act, int ld_act, const uint16_t* wp_down, int64_t expert_stride_bytes,
                           int n_experts, int d, int hidden, int k, const int32_t* offsets, const int32_t* pair_of,
                           const uint16_t* expert_w, uint16_t* y, int ldy, void* stream);
/* The same two for n_pairs pairs whose number the host knows: from 12 pairs an expert on, in tiles of an expert's pairs. */
int ohara_moe_experts_gate_up_many(const uint16_t* x, int ldx, const uint16_t* wp_gate_up, int64_t expert_stride_bytes,
                                   int n_experts, int hidden, int d, int k, int n_pairs, const int32_t* offsets,
                                   const int32_t* pair_of, uint16_t* act, int ld_act, void* stream);
int ohara_moe_experts_down_many(const uint16_t* act, int ld_act, const uint16_t* wp_down, int64_t expert_stride_bytes, int n_experts,
                                int d, int hidden, int k, int n_pairs, const int32_t* offsets, const int32_t* pair_of,
                                const uint16_t* expert_w, uint16_t* y, int ldy, void* stream);
int ohara_moe_combine(const uint16_t* y, int ldy, const int32_t* expert_idx, const int32_t* pos_of, int n_tokens, int k,
                      const uint16_t* shared, int ld_shared, const uint16_t* resid, int ldr, uint16_t* out, int ldo, int d,
                      void* stream);
/* The same feed-forward for a decode step in four launches (at most 64 experts, 1024 pairs, d <= 4096):
 *  ohara_moe_route_fused    the block's RMSNorm (ohara/modules/norm.py:16-21; ohara/models/llama.py:200) of the rows
 *                           x, the router Linear on the normalised rows (moe_grouped.py:126), _route (:122-147) and
 *                           the sort of :161-168 in ONE launch: x_norm (n_tokens, d) for the experts, expert_idx /
 *                           expert_w, offsets / pair_of / pos_of as above; router_logits (n_tokens, n_experts) may be
 *                           NULL.  counter: one int32 of device memory that is zero between calls (the workgroup
 *                           that finishes last sorts, and leaves it zero); calls that share it must not overlap.
 *  ohara_moe_experts_gate_up_shared / ohara_moe_experts_down_shared
 *                           the expert launches with the shared expert (_shared, :206-207, 219-220) as more
 *                           rows of their grids (16 tokens a row): wp_shared its packed gate/up (down) rows, shared_hidden its width,
 *                           act_shared (n_tokens, shared_hidden), y_shared (n_tokens, d) = bf16(act_shared W_down),
 *                           not scaled - pass y_shared to ohara_moe_combine as `shared`.  wp_shared NULL: as the
 *                           entry points above. */
int ohara_moe_route_fused(const uint16_t* x, int ldx, const uint16_t* norm_w, float eps, const uint16_t* router_wp,
                          const uint16_t* router_bias, int n_tokens, int d, int n_experts, int k, int biased_topk,
                          int gate_sigmoid, int normalize, uint16_t* x_norm, int ld_x_norm, uint16_t* router_logits, int ldl,
                          int32_t* expert_idx, uint16_t* expert_w, int32_t* offsets, int32_t* pair_of, int32_t* pos_of,
                          int32_t* counter, void* stream);
int ohara_moe_experts_gate_up_shared(const uint16_t* x, int ldx, const uint16_t* wp_gate_up, int64_t expert_stride_bytes,
                                     int n_experts, int hidden, int d, int k, const int32_t* offsets,
                                     const int32_t* pair_of, uint16_t* act, int ld_act, const uint16_t* wp_shared,
                                     int shared_hidden, int n_tokens, uint16_t* act_shared, int ld_act_shared,
                                     void* stream);
int ohara_moe_experts_down_shared(const uint16_t* act, int ld_act, const uint16_t* wp_down, int64_t expert_stride_bytes,
                                  int n_experts, int d, int hidden, int k, const int32_t* offsets, const int32_t* pair_of,
                                  const uint16_t* expert_w, uint16_t* y, int ldy, const uint16_t* wp_shared,
                                  int shared_hidden, int n_tokens, const uint16_t* act_shared, int ld_act_shared,
                                  uint16_t* y_shared, int ldy_shared, void* stream);

/* ---- the whole forward pass through the KV cache ---------------------------------
 * Llama.forward(x, kv_cache, position) (ohara/models/llama.py:279-323; Block.forward
 * :191-201) for seq_len new tokens per sequence, as a fixed sequence of the kernels
 * above enqueued on `stream`; optionally followed by greedy selection that feeds the
 * next call, so a generate loop (ohara/chat_engine.py:395-405,
 * ohara/inference.py:110-121) can run without touching the host.
 * Host structs; every pointer inside is a device pointer owned by the caller. */
typedef struct OharaLayer {
  const uint16_t* wqkv;  /* packed rows [W_q; W_k; W_v], each (heads*dh, d)          */
  const uint16_t* wo;    /* packed attn.proj (d, h*dh)                                */
  const uint16_t* wgu;   /* packed ff.gate / ff.up, rows interleaved (swiglu perm)    */
  const uint16_t* wdown; /* packed ff.down (d, f)                                     */
  const uint16_t* norm1; /* (d) */
  const uint16_t* norm2; /* (d) */
} OharaLayer;

typedef struct OharaModel {
  int32_t n_layers, d_model, n_heads, n_kv_heads, head_dim, d_ff, vocab, t_max;
  float eps;
  int32_t reserved;
  const uint16_t* token_emb;  /* (vocab, d) row-major, unpacked */
  const uint16_t* final_norm; /* (d) */
  const uint16_t* w_vocab;    /* packed vocab_proj (vocab, d) */
  const uint16_t* cos;        /* (2*t_max, dh/2) bf16 */
  const uint16_t* sin;
  const OharaLayer* layers;   /* host array [n_layers] */
} OharaModel;

typedef struct OharaDecodeState {
  int32_t batch;         /* sequences                                                     */
  int32_t rows_cap;      /* rows (batch*seq_len) the activation buffers below can hold    */
  int32_t n_split;       /* context chunks of decode attention (seq_len == 1)             */
  int32_t valid_vocab;   /* ids >= this are never selected; 0 = whole vocabulary          */
  int32_t hist_cap;
  int32_t prof_kernel;   /* -1: off; else index of the launch (0 = embedding, 1 + 5*l + i = i-th
                            kernel of layer l, 1 + 5*n_layers = vocabulary projection, then the
                            selection) to bracket with prof_start / prof_stop                    */
  int64_t* ids;          /* (rows) tokens fed; ids[0:batch] overwritten by greedy select  */
  uint16_t* x;           /* (rows, d) residual stream                                     */
  uint16_t* q;           /* (rows, h*dh)                                                  */
  uint16_t* attn;        /* (rows, h*dh)                                                  */
  uint16_t* act;         /* (rows, f)                                                     */
  uint16_t* xn;          /* (rows, d) normalised rows for calls with > 64 rows (> 32 where d > 1024, > 16
                            where d > 2048); may be NULL (the skinny kernel then norms the rows itself, 64 at a
                            time, instead of the tiled MFMA kernel)                            */
  uint16_t* logits;      /* (batch, vocab) or (rows, vocab), see logits_mode              */
  void* attn_ws;         /* ohara_attn_workspace_bytes(batch, h, h_kv, dh, n_split); calls with
                            seq_len > 1 keep partial results there (ohara_attn_prefill_ws_bytes)
                            where the room behind its counters, align256(4 batch h_kv) bytes, is enough */
  int32_t* step_state;   /* 4 x int32 {pos, step, done, pad}, may be NULL                 */
  int64_t* history;      /* (hist_cap, batch) generated ids, may be NULL                  */
  uint16_t* const* kcache; /* host array [n_layers] of (batch_cap, t_max, h_kv, dh)       */
  uint16_t* const* vcache;
  /* int8 cache mode (kv_int8 != 0): kcache / vcache point at int8 tensors of the same shape,
     kvstats at the per-layer (batch_cap, h_kv, t_max, 4) fp32 statistics records; kstage / vstage
     (rows, h_kv*dh) receive the bf16 rows before they are quantised; kdeq / vdeq ((batch, t_max,
     h_kv, dh) bf16, may be NULL) hold the dequantised cache for calls with >= 16 positions. */
  int32_t kv_int8;
  float* const* kvstats;
  uint16_t* kstage;
  uint16_t* vstage;
  uint16_t* kdeq;
  uint16_t* vdeq;
  /* ragged batches: when non-NULL, sequence b's first fed token sits at cache position seq_pos[b]
     (device array of `batch` entries) and the pos / use_pos_dev arguments are ignored.  The
     reference has one scalar position for the whole batch (llama.py:287-299); this is what lets
     sequences of different lengths decode in one batch.  bf16 caches only. */
  const int32_t* seq_pos;
  void* prof_start;      /* hipEvent_t recorded on `stream` right before launch prof_kernel */
  void* prof_stop;       /* hipEvent_t recorded right after it                             */
} OharaDecodeState;

#define OHARA_LOGITS_NONE 0
#define OHARA_LOGITS_LAST 1 /* logits (batch, vocab) of each sequence's last position     */
#define OHARA_LOGITS_ALL 2  /* logits (batch*seq_len, vocab), what llama.py:321-322 returns */

/* pos: cache position of the first fed token (ignored when use_pos_dev != 0, then
 * step_state->pos is read on the device; that needs seq_len == 1).
 * select_greedy != 0 (needs logits_mode LAST or seq_len == 1) appends the argmax. */
int ohara_llama_forward(const OharaModel* m, const OharaDecodeState* s, int seq_len, int pos, int use_pos_dev,
                        int logits_mode, int select_greedy, void* stream);

/* The same for a model whose feed-forwards are grouped experts (moe_grouped.py:209-228) or dense, over caches of bfloat16 or int8.
 * `scratch`: ohara_moe_forward_bytes of the same arguments, 256-byte aligned, used by this call alone; attn_ws:
 * ohara_attn_workspace_bytes(batch, h, h_kv, dh, n_split), zero between calls.  logits: (batch, vocab) of the last tokens, or
 * (batch * seq_len, vocab). */
typedef struct OharaMoeLayer {
  const uint16_t *wqkv, *wo, *norm1, *norm2;
  const uint16_t *wgu, *wdown;               /* packed: the dense feed-forward's, or the shared expert's (NULL: none), ff wide */
  const uint16_t *router, *router_bias;      /* router NULL: a dense layer                       */
  const uint16_t *experts_gu, *experts_down; /* as ohara_moe_experts_gate_up_shared / _down_shared */
  int64_t gu_stride, down_stride;            /* bytes from expert to expert                      */
  int32_t* counter;
  int32_t ff, n_experts, hidden, k, biased_topk, gate_sigmoid, normalize, reserved;
} OharaMoeLayer;

typedef struct OharaMoeCall {
  int32_t n_layers, d_model, n_heads, n_kv_heads, head_dim, vocab, t_max;
  int32_t batch, seq_len, pos, n_split, last_only;
  float eps;
  int32_t reserved;
  const uint16_t *token_emb, *final_norm, *w_vocab, *cos, *sin;
  const OharaMoeLayer* layers;               /* host array [n_layers]                            */
  const int64_t* ids;                        /* (batch, seq_len)                                 */
  void* const* kcache;                       /* host arrays [n_layers]                           */
  void* const* vcache;
  void* const* kvstats;                      /* int8 caches; NULL: bfloat16                      */
  uint16_t* logits;
  void *attn_ws, *scratch;
  int64_t scratch_bytes;
} OharaMoeCall;

int64_t ohara_moe_forward_bytes(const OharaMoeCall* c);
int ohara_moe_forward(const OharaMoeCall* c, void* stream);

/* ohara_llama_forward over n prompts of different lengths, each from position 0 into its own row of the caches (bf16 caches,
 * head width 64 or 128); logits (n, vocab) of the last token of each.  s: ids, x, xn, q, attn and act for the rows of all prompts
 * side by side.  `lengths` on the host; `table` on the device: n first rows, n lengths, n rows of the caches, then the position of
 * every row and the row of the caches it belongs to. */
int ohara_llama_prompts(const OharaModel* m, const OharaDecodeState* s, int n, const int32_t* lengths, const int32_t* table,
                        void* stream);


/* ---- one decode step as ONE persistent launch (batch <= 16) ------------------------
 * Same result as ohara_llama_forward(seq_len = 1, use_pos_dev = 1, LOGITS_LAST) but the
 * whole step (all layers, vocabulary projection, greedy selection) runs in a single
 * kernel of `n_workgroups` resident workgroups (use the CU count; more than the device can
 * hold of this kernel at once returns OHARA_ESIZE) whose phases are separated by grid-wide barriers
 * (batch > 8) or hand their rows over through memory that the consumers poll (batch <= 8); it has no counterpart in the reference, whose decode step is
 * ~1000 eager launches (llama.py:279-323).  The cache position and step index are read
 * from / advanced in s->step_state; s->attn and s->attn_ws are not used.
 * `workspace`: ohara_persistent_workspace_bytes(m, batch, s->n_split, n_workgroups) of
 * device memory with any contents (it need not be zeroed: the call with init_workspace = 1 sets
 * what a step relies on, every other slot a step reads was written earlier in the same step, and
 * the merge of the attention chunks never uses a chunk no workgroup wrote).  Call once with
 * init_workspace = 1 (copies the layer table and the cache pointers to the device, zeroes the
 * barrier words and the launch counters and fills the hand-off rows and the attention partials of the
 * polled builds (batch <= 8) with 0xFF, their "not written yet"; synchronises the stream;
 * do it outside graph capture) whenever the model or the caches change, and before the workspace
 * is used for the first time or after its memory has been used for anything else; then each call
 * with init_workspace = 0 enqueues one step.  Steps on one workspace must not overlap (each
 * step counts itself in the workspace).  spin_limit bounds every barrier wait and every poll for
 * a hand-off (0 = default); if a wait expires the kernel still drains and the error word reads
 * non-zero.  s->n_split must be 16.
 * Requires head_dim 64 or 128, n_heads / n_kv_heads in {1, 2, 4}, d_model <= 1024,
 * d_model and d_ff multiples of 8. */
int64_t ohara_persistent_workspace_bytes(const OharaModel* m, int batch, int n_split, int n_workgroups);
int ohara_llama_decode_persistent(const OharaModel* m, const OharaDecodeState* s, void* workspace, int n_workgroups,
                                  int init_workspace, int select_greedy, unsigned int spin_limit, void* stream);
/* Byte offsets inside the workspace: the barrier words; the sticky error word (uint32,
 * non-zero after a barrier wait expired); per workgroup 1024 x uint64 samples of the constant
 * 100 MHz clock taken by its thread 0 at every phase boundary when s->prof_kernel == -2 (workgroup
 * w's samples start 8192 w bytes after the offset; measurement only; the samples
 * are compiled into a separate build of the kernel that exists for head_dim 128 with
 * n_kv_heads == n_heads only, other shapes leave the slots untouched). */
int64_t ohara_persistent_barrier_offset(const OharaModel* m, int batch, int n_split, int n_workgroups);
/* Which build of the kernel a launch with this model, batch and grid runs: 0 the general one (a grid
 * barrier between the phases), 1 and 2 the polled ones (one sequence; two to eight).  The polled builds
 * also serve the int8 cache (s->kv_int8: the attention phase dequantises the tiles it reads and
 * quantises the appended row as ohara_kv_quant_append_int8 does, ohara/modules/kv_cache.py:15-32);
 * ohara_llama_decode_persistent returns OHARA_ESIZE for an int8 cache where this returns 0. */
int ohara_persistent_polled(const OharaModel* m, int batch, int n_workgroups);
int64_t ohara_persistent_error_offset(const OharaModel* m, int batch, int n_split, int n_workgroups);
int64_t ohara_persistent_profile_offset(const OharaModel* m, int batch, int n_split, int n_workgroups);

/* ---- one decode step of the BitNet-b1.58 Llama as ONE persistent launch (batch <= 8) --------
 * Llama.forward(x, kv_cache, position) (ohara/models/llama.py:279-323) for one new token per
 * sequence when the seven projections of every block are BitLinears
 * (experiments/bitnet/bitnet.py:29-95, swapped in by apply_bitlinear :70-95 over the target list of
 * experiments/bitnet/train_bitnet.py:240): per projection the BitLinear's own RMSNorm, the
 * per-token int8 codes, the ternary product on the integer matrix cores and the rescale; block
 * norms, rotary, cache append, attention, SwiGLU, residuals, the final norm, the bf16 vocabulary
 * projection and the greedy selection as in ohara_llama_decode_persistent, whose calling
 * convention (init_workspace, step_state, spin_limit, error word) this entry point shares.  The
 * integer accumulators are those of ohara_bitlinear_* on the same rows; the reference's eager
 * step is ~1700 launches.
 * w[i] / norm_w[i] / gamma[i]: packed ternary weight (ohara_bitlinear_pack_ternary), the
 * BitLinear's norm weight and weight scale of attn.query, attn.key, attn.value, attn.proj,
 * ff.gate, ff.up, ff.down in that order.
 * Requires head_dim 64 or 128, n_heads == n_kv_heads, d_model and n_heads * head_dim <= 2048,
 * d_ff <= 6144, d_model and d_ff multiples of 16, n_workgroups >= 4; s->n_split must be 16; uses s->batch, valid_vocab, hist_cap, ids, logits,
 * step_state, history, kcache, vcache. */
#define OHARA_BIT_QUERY 0
#define OHARA_BIT_KEY 1
#define OHARA_BIT_VALUE 2
#define OHARA_BIT_PROJ 3
#define OHARA_BIT_GATE 4
#define OHARA_BIT_UP 5
#define OHARA_BIT_DOWN 6
typedef struct OharaBitLayer {
  const uint32_t* w[7];
  const uint16_t* norm_w[7];
  float gamma[7];
  float reserved;
  const uint16_t* norm1; /* (d) block norms */
  const uint16_t* norm2;
} OharaBitLayer;

typedef struct OharaBitModel {
  int32_t n_layers, d_model, n_heads, n_kv_heads, head_dim, d_ff, vocab, t_max;
  float eps;
  int32_t reserved;
  const uint16_t* token_emb;  /* (vocab, d) row-major, unpacked */
  const uint16_t* final_norm; /* (d) */
  const uint16_t* w_vocab;    /* packed vocab_proj (vocab, d), bf16 (ohara_pack_rows_bf16) */
  const uint16_t* cos;        /* (2*t_max, dh/2) bf16 */
  const uint16_t* sin;
  const OharaBitLayer* layers; /* host array [n_layers] */
} OharaBitModel;

int64_t ohara_bitnet_persistent_workspace_bytes(const OharaBitModel* m, int batch, int n_workgroups);
int64_t ohara_bitnet_persistent_error_offset(const OharaBitModel* m, int batch, int n_workgroups);
/* 1024 x uint64 shader-clock samples of workgroup 0 (six per grid barrier: phase work issued, own
 * stores complete, workgroup barrier passed, arrival issued, prefetch issued, barrier passed; a single
 * sequence: ten per layer, behind every poll and phase, and those of the down projection's first
 * workgroup 512 words on), taken
 * when s->prof_kernel == -2 (measurement only; a separate build of the kernel that exists for
 * head_dim 128 only, other shapes leave the slots untouched). */
int64_t ohara_bitnet_persistent_profile_offset(const OharaBitModel* m, int batch, int n_workgroups);
int ohara_bitnet_decode_persistent(const OharaBitModel* m, const OharaDecodeState* s, void* workspace, int n_workgroups,
                                   int init_workspace, int select_greedy, unsigned int spin_limit, void* stream);

/* ---- Phi (ohara/models/phi.py): the parts of its cached decode path that differ from Llama ----
 * nn.Linear WITH bias on packed weights (phi.py:46-47, :63-66, :161), any number of rows (up to 64,
 * or 16 where k > 1024: the weight-streaming strip kernel; more: the tiled MFMA kernel of ohara_gemm_bf16,
 * same epilogues and rounding points).  n % 4 == 0, k % 8 == 0.
 *   OHARA_LIN_BIAS       out = bf16(x @ W^T + bias)
 *   OHARA_LIN_BIAS_GELU  out = new_gelu(bf16(x @ W^T + bias)), every op of phi.py:37-40 rounded to
 *                        bf16 as the eager ops round                          (MLP.fc1, phi.py:50-51)
 *   OHARA_LIN_BIAS_ADD2  out = bf16(bf16(add1 + bf16(x @ W^T + bias)) + add2): the parallel block's
 *                        `mixer(x) + mlp(x) + residual` with add1 = mixer output, add2 = block input
 *                                                                              (phi.py:151) */
#define OHARA_LIN_BIAS 0
#define OHARA_LIN_BIAS_GELU 1
#define OHARA_LIN_BIAS_ADD2 2
int ohara_linear_bias_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, int rows,
                           int epilogue, const uint16_t* add1, int ld1, const uint16_t* add2, int ld2, uint16_t* out,
                           int ldo, void* stream);
/* OHARA_LIN_BIAS_ADD2 with room (16-byte aligned, _bytes; 0: none needed) for a product in parts of its depth, where rows are too few to
 * keep the CUs busy over all of it.  Too little room or NULL: as without. */
int64_t ohara_linear_bias_add2_bytes(int rows, int n, int k);
int ohara_linear_bias_add2_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, int rows, const uint16_t* add1,
                                int ld1, const uint16_t* add2, int ld2, uint16_t* out, int ldo, void* workspace, int64_t workspace_bytes, void* stream);
/* resid (rows, n) += x W^T, then, where norm_w is given, xn = its RMSNorm (ohara_rmsnorm_bf16); room as above. */
int64_t ohara_gemm_residual_norm_bytes(int rows, int n, int k);
int ohara_gemm_residual_norm_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, int rows, uint16_t* resid, const uint16_t* norm_w,
                                  float eps, uint16_t* xn, void* workspace, int64_t workspace_bytes, void* stream);
/* The head of a Phi block in one launch (phi.py:150, :81-87, :95, :50-51): h = LayerNorm(x), then
 * [q; k; v; fc1] = h @ W^T + bias with W the packed vertical concatenation of q_proj, k_proj, v_proj
 * (d rows each) and mlp.fc1 (ff rows): q rows -> q (leading dimension ldq), k / v rows -> the
 * caches at position pos + s as they are (un-rotated), fc1 rows -> new_gelu -> act.  Same rounding
 * points as ohara_layernorm_bf16 + ohara_linear_bias_bf16 + ohara_kv_append_bf16, except that the
 * variance comes from the sums of x and x^2 where ohara_phi_block_norms is 0.  ln_w == NULL: x already is
 * the normalised input (there a separate LayerNorm launch costs less than re-deriving the statistics
 * in every workgroup before its weight loads start).
 * d % 16 == 0, ff % 4 == 0. */
int ohara_phi_block_in_bf16(const uint16_t* x, int ldx, const uint16_t* ln_w, const uint16_t* ln_b, float eps,
                            const uint16_t* wp, const uint16_t* bias, int d, int ff, int batch, int seq_len, int pos,
                            const int32_t* pos_dev, uint16_t* q, int ldq, uint16_t* kcache, uint16_t* vcache, int t_max,
                            uint16_t* act, int ldact, void* stream);
/* 1 where that call, given ln_w, is quicker than with a launch of ohara_layernorm_bf16 ahead of it (the same bits). */
int ohara_phi_block_norms(int rows, int d, int ff);
/* nn.LayerNorm over the last dimension (phi.py:132, :160): fp32 mean and biased variance,
 * out = bf16((x - mean) * rstd * weight + bias).  d % 8 == 0. */
int ohara_layernorm_bf16(const uint16_t* x, int ldx, const uint16_t* weight, const uint16_t* bias, uint16_t* out, int ldo,
                         int rows, int d, float eps, void* stream);
/* KVCache.forward for rows that are stored as they are (phi.py:95, kv_cache.py:104-105): row
 * (b, s) of k / v (leading dimension ld, h*dh wide) -> cache[b, pos + s].  pos_dev (seq_len 1):
 * the position is read on the device. */
int ohara_kv_append_bf16(const uint16_t* k, const uint16_t* v, int ld, int batch, int seq_len, int h, int dh, int pos,
                         const int32_t* pos_dev, uint16_t* kcache, uint16_t* vcache, int t_max, void* stream);
/* PhiMHA's attention core (phi.py:98-117): fp32 throughout; the first `rot` features of every head
 * rotate in the half-split layout (feature i with i + rot/2; rotary.py:131-164), queries from
 * position pos (+ s), the cached UN-rotated keys from 0; key t is visible to query s when
 * t <= pos + s; softmax(q k^T / sqrt(dh)) v rounded once to bf16.  cos / sin: (t_max, rot/2) fp32
 * tables of rotary.py:166-184.  q: rows (b, s) with leading dimension ldq; out (batch*seq_len, h*dh).
 * dh % 8 == 0, dh <= 128.  n_split > 1 (seq_len 1 only, at most 64) spreads the context of every
 * (sequence, head) over that many workgroups whose partial results meet in `workspace`
 * (ohara_phi_attn_workspace_bytes, zero-filled once before the first use; calls sharing it must not
 * overlap) and are merged in chunk order by the workgroup that finishes last.  Calls with 16 or more
 * new tokens per sequence (prefill; head widths 16, 32, 64, 80, 128) run queries in tiles of 64
 * against key / value tiles in LDS with fp32 matrix products; other shapes one query per workgroup. */
int64_t ohara_phi_attn_workspace_bytes(int batch, int h, int dh, int n_split);
int ohara_phi_attn_bf16(const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos,
                        const float* sin, int rot, int batch, int seq_len, int h, int dh, int t_max, int pos,
                        const int32_t* pos_dev, int n_split, void* workspace, uint16_t* out, void* stream);
// In how many teams of waves a workgroup of such a prefill shares its queries' positions (rotated features in eights).
int ohara_phi_prefill_teams(int batch, int seq_len, int h, int pos);
// The same for one token a sequence, and beside it a product that does not wait for it: y = x W^T + bias as ohara_linear_bias_bf16 gives it,
// x (batch, k), y (batch, n).  Neither may read what the other writes.  Where pos_dev is given, `pos` is about
// where it will be: how far back the attention goes decides whether one launch or two are quicker.
int ohara_phi_attn_linear_bf16(const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos, const float* sin, int rot,
                               int batch, int h, int dh, int t_max, int pos, const int32_t* pos_dev, int n_split, void* workspace, uint16_t* out,
                               const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, uint16_t* y, int ldy, void* stream);

// Into how many chunks that cuts the context where one launch does both; 0 where it makes two launches (as it also does where an angle's eighths do
// not lie on 16 bytes or inside one half of the rotated features).
int ohara_phi_attn_linear_chunks(int batch, int h, int dh, int n_split, int pos, int n, int k);

// Both, and behind them the attention's output projection with its bias and two addends: out = bf16(bf16(y + attention W_out^T + bias_out) + add), W_out
// (n, h * dh), add and out (batch, n).  The projection's launch merges the attention's chunks, which spares that the wait for the last of them.  They are
// added up by fours first: of the attention's values up to 9 in 100 000 round to another bf16 number than those of ohara_phi_attn_bf16 over as many chunks (20 to 28 of
// either are not the rounded ones of 64 bits, behind 100 to 1100 positions).  The products' bits are those of ohara_linear_bias_bf16.  The workspace is
// ohara_phi_attn_bf16's, on 16 bytes.
int ohara_phi_attn_out_bf16(const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos, const float* sin, int rot,
                            int batch, int h, int dh, int t_max, int pos, const int32_t* pos_dev, int n_split, void* workspace, const uint16_t* x, int ldx,
                            const uint16_t* wp, int n, int k, const uint16_t* bias, uint16_t* y, int ldy, const uint16_t* wp_out, const uint16_t* bias_out,
                            const uint16_t* add, int ld_add, uint16_t* out, int ldo, void* stream);
// Chunks of a context at most in that call; 0 where it is refused (OHARA_ESIZE): where the calls above are the quicker ones, or its kernels don't fit.
int ohara_phi_attn_out_chunks(int batch, int h, int dh, int rot, int n_split, int pos, int n, int k);

/* ---- hybrid decoders: attention with a distance bias beside recurrent layers -----------------------
 * (no counterpart in the reference.)  Entry points ending in _bf16 keep activations, caches and weights
 * in bfloat16, those ending in _f32 in 32-bit floats; the residual stream, every norm, score, softmax
 * weight, decay and recurrent state is fp32 in both.  Vectors (norm, convolution, decay parameters)
 * are fp32 in both.
 *
 * OharaSeq says which rows of a call belong to which sequence and where they sit: the call has
 * batch * seq_len rows ordered (sequence, token); token s of sequence b sits at position start(b) + s with
 * start(b) = pos, *pos_dev or pos_dev[b] (pos_stride 0 / 1).  lens: tokens of each sequence in this call
 * (rows past them are padding: they change no cache or state and their results mean nothing); NULL: all
 * have seq_len.  slots: cache row of each sequence; NULL: sequence b uses row b.  Two sequences of a call
 * never share a cache row. */
typedef struct OharaSeq {
  int batch, seq_len, pos, pos_stride;
  const int32_t* pos_dev;
  const int32_t* lens;
  const int32_t* slots;
} OharaSeq;

/* What the residual kernel puts into `out` after updating the residual row x. */
#define OHARA_OUT_NONE 0
#define OHARA_OUT_COPY 1 /* x */
#define OHARA_OUT_CONV 2 /* x + causal depthwise convolution of x over time (seq_len 1; see conv_w / ring) */
#define OHARA_OUT_NORM 3 /* group RMS norm of x times norm2_w */
/* May be added to out_mode (groups 1 only): the norm of y / of OHARA_OUT_NORM is a layer norm without bias,
 * i.e. the row's mean is taken off before the root mean square. */
#define OHARA_CENTER_Y 16
#define OHARA_CENTER_OUT 32

/* Output of routed experts before it is summed: row n of the layer's output is
 *   sum_j w[n*top + j] * (idx[n*top + j] < experts ? y[pos_of[n*top + j]] : h[n]) + shared[n]   (shared: NULL for none),
 * in fp32 and in the order of j (w NULL: all weights are 1); rows of y, h, shared in the activation type, leading dimensions multiples of 4. */
typedef struct OharaMixture {
  int top, experts, ldy, ldh, lds, reserved;
  const float* w;
  const int32_t* idx;
  const int32_t* pos_of;
  const void* y;
  const void* h;
  const void* shared;
} OharaMixture;

/* Residual update of a block with norms on the sublayer outputs, one launch:
 *   ids != NULL:  x = table_scale * table[id] (table: activation type, vocab rows of d)
 *   y != NULL:    x += norm_w * group_rms(y)  (groups equal runs of the row, each over sqrt(mean square + eps))
 *   mix != NULL:  the same with the rows of an OharaMixture as y
 *   norm_w NULL:  x += y, without a norm
 * x: (rows, d) fp32, updated in place.  out (leading dimension ldo >= d, columns past d are set to zero)
 * per out_mode.  OHARA_OUT_CONV: conv_w (taps, d) fp32 with the current token's row last, ring
 * (cache rows, taps, d) fp32 holds the inputs of the last tokens at index position mod taps and is
 * updated; inputs before position 0 count as zero, so a ring needs no clearing when its row is reused.
 * OHARA_OUT_NORM takes norm2_w. */
int ohara_residual_norm_bf16(float* x, int d, const int64_t* ids, const uint16_t* table, int vocab, float table_scale, const uint16_t* y,
                             int ldy, const float* norm_w, int groups, float eps, int out_mode, uint16_t* out, int ldo,
                             const float* norm2_w, const float* conv_w, int taps, float* ring, const OharaMixture* mix, const OharaSeq* seq,
                             void* stream);
int ohara_residual_norm_f32(float* x, int d, const int64_t* ids, const float* table, int vocab, float table_scale, const float* y, int ldy,
                            const float* norm_w, int groups, float eps, int out_mode, float* out, int ldo,
                            const float* norm2_w, const float* conv_w, int taps, float* ring, const OharaMixture* mix, const OharaSeq* seq,
                            void* stream);
/* out = x + causal depthwise convolution of x over time for any seq_len (the ring is only read: follow with
 * ohara_conv_ring_store_f32), columns d .. ldo-1 of out are set to zero. */
int ohara_input_conv_bf16(const float* x, int d, const float* conv_w, int taps, const float* ring, uint16_t* out, int ldo,
                          const OharaSeq* seq, void* stream);
int ohara_input_conv_f32(const float* x, int d, const float* conv_w, int taps, const float* ring, float* out, int ldo,
                         const OharaSeq* seq, void* stream);
/* The last taps - 1 input rows of each sequence (src: rows of `channels`, leading dimension ld) -> ring
 * (cache rows, taps, channels) at index position mod taps. */
int ohara_conv_ring_store_bf16(const uint16_t* src, int ld, int channels, int taps, uint16_t* ring, const OharaSeq* seq,
                               void* stream);
int ohara_conv_ring_store_f32(const float* src, int ld, int channels, int taps, float* ring, const OharaSeq* seq,
                              void* stream);

/* Plain fp32 product for models served in 32-bit: y = x W^T (+ bias), W (n, k) fp32 row-major, k % 4 == 0.
 * w_up != NULL: y = silu(x W^T) * (x w_up^T).  cap > 0: y = cap * tanh(y / cap). */
int ohara_gemm_f32(const float* x, int ldx, const float* w, const float* w_up, const float* bias, float cap, int n, int k,
                   int rows, float* out, int ldo, void* stream);
/* ohara_gemm_skinny_bf16 without a norm and with y = bf16(cap * tanh(fp32 sum / cap)) as the epilogue
 * (vocabulary projections with soft-capped logits). */
int ohara_gemm_softcap_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, float cap, int rows,
                            uint16_t* out, int ldo, void* stream);

/* Two-sided activation with fixed coefficients, f(z) = z / 2 + above z^2 for z > 0, z / 2 + below (exp(z) - 1 - z) for z <= 0, of
 * z = x W^T + bias in fp32 (n, ldo and the bias as ohara_linear_bias_bf16 / ohara_gemm_f32). */
int ohara_gemm_xielu_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, float above, float below,
                          int rows, uint16_t* out, int ldo, void* stream);
int ohara_gemm_xielu_f32(const float* x, int ldx, const float* w, int n, int k, const float* bias, float above, float below, int rows,
                         float* out, int ldo, void* stream);

/* Constants of a clamped gated unit. */
typedef struct OharaGlu {
  float limit, alpha, offset;
  int reserved;
} OharaGlu;
/* Clamped gated unit: out = g sigmoid(alpha g) (u + offset), g = min(x Wg^T, limit), u = min(max(x Wu^T, -limit), limit), in fp32 up
 * to the store.  bf16: packed weight in the order of ohara_swiglu_perm, any rows; f32: two matrices (n, k) row-major. */
int ohara_gemm_glu_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, float limit, float alpha, float offset,
                        int rows, uint16_t* out, int ldo, void* stream);
int ohara_gemm_glu_f32(const float* x, int ldx, const float* w_gate, const float* w_up, int n, int k, float limit, float alpha,
                       float offset, int rows, float* out, int ldo, void* stream);

/* out[row, i] = gelu_tanh((x W^T)[row, i]) * table[ids[row] * ldt + i], gelu_tanh(z) = z/2 (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))),
 * i < n: a projection gated onto an embedding of the row's token (table: rows of ldt entries, the layer's n from the pointer on).
 * The sum stays fp32 up to the product.  bf16: packed weight, n and ldt multiples of 4, any rows; f32: W (n, k) row-major. */
int ohara_gemm_gelu_lookup_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* table, int ldt,
                                const int64_t* ids, int vocab, int rows, uint16_t* out, int ldo, void* stream);
int ohara_gemm_gelu_lookup_f32(const float* x, int ldx, const float* w, int n, int k, const float* table, int ldt,
                               const int64_t* ids, int vocab, int rows, float* out, int ldo, void* stream);

/* A layer's side embedding with the residual updates on either side, one launch (every norm over the whole row with eps):
 *   x += norm_w * norm(y);  z = gelu_tanh(Wg x) * table[ids[row] * ldt + i];  x += side_w * rms(Wp z);  out = out_w * norm(x)
 * x: (rows, d) fp32, updated in place; y: rows of ldy; gate, proj: packed Wg (n, d rounded up to 8) and Wp (d rounded up to 8, n);
 * center_y / center_out: that norm is a layer norm without bias.  d, ldy and ldo multiples of 4, n <= 256.  x, z and Wp z are
 * rounded to bf16 for the products.  rows_per_group: rows of a workgroup (a power of two up to 16), rows_per_group * d <= 16384. */
int ohara_token_side_bf16(float* x, int d, const uint16_t* y, int ldy, const float* norm_w, int center_y, const uint16_t* gate,
                          const uint16_t* proj, int n, const uint16_t* table, int ldt, const int64_t* ids, int vocab,
                          const float* side_w, float eps, const float* out_w, int center_out, int rows, int rows_per_group,
                          uint16_t* out, int ldo, void* stream);

/* Attention front end off one projection p with row layout [q (h*dh); k (h_kv*dh); v (h_kv*dv); ...]:
 * q and k are each divided by the root mean square of ALL their elements of the row and multiplied by
 * qn / kn; every value head is divided by its own root mean square.  q -> q_out (rows, h, dhp), keys and
 * values -> caches (cache rows, t_max, h_kv, dhp) and (.., dvp) at the tokens' positions; dhp / dvp are
 * dh / dv rounded up to multiples of 8, the columns past dh / dv are set to zero. */
int ohara_qkv_norm_append_bf16(const uint16_t* p, int ldp, int h, int h_kv, int dh, int dv, const float* qn,
                               const float* kn, float eps, uint16_t* q_out, uint16_t* kcache, uint16_t* vcache, int t_max,
                               const OharaSeq* seq, void* stream);
int ohara_qkv_norm_append_f32(const float* p, int ldp, int h, int h_kv, int dh, int dv, const float* qn, const float* kn,
                              float eps, float* q_out, float* kcache, float* vcache, int t_max, const OharaSeq* seq,
                              void* stream);
/* The same layout without norms: the first rot dimensions of every q and k head are rotated in neighbouring pairs,
 * (u, v) -> (u cos - v sin, v cos + u sin) with the angles' tables cos, sin (t_max, rot / 2) fp32 at the token's position. */
int ohara_qkv_rotate_append_bf16(const uint16_t* p, int ldp, int h, int h_kv, int dh, int dv, const float* cos,
                                 const float* sin, int rot, uint16_t* q_out, uint16_t* kcache, uint16_t* vcache, int t_max,
                                 const OharaSeq* seq, void* stream);
int ohara_qkv_rotate_append_f32(const float* p, int ldp, int h, int h_kv, int dh, int dv, const float* cos, const float* sin,
                                int rot, float* q_out, float* kcache, float* vcache, int t_max, const OharaSeq* seq,
                                void* stream);
/* The same with every q and k head first divided by its own root mean square and multiplied by qn / kn (dh entries, shared by
 * the heads).  dh, dv <= 256. */
int ohara_qkv_headnorm_rotate_append_bf16(const uint16_t* p, int ldp, int h, int h_kv, int dh, int dv, const float* qn,
                                          const float* kn, float eps, const float* cos, const float* sin, int rot,
                                          uint16_t* q_out, uint16_t* kcache, uint16_t* vcache, int t_max, const OharaSeq* seq,
                                          void* stream);
int ohara_qkv_headnorm_rotate_append_f32(const float* p, int ldp, int h, int h_kv, int dh, int dv, const float* qn,
                                         const float* kn, float eps, const float* cos, const float* sin, int rot, float* q_out,
                                         float* kcache, float* vcache, int t_max, const OharaSeq* seq, void* stream);
/* Causal attention over the cache with a linear distance bias and a per-head output gate:
 *   o[row, hd, :] = sigmoid(gate[row, hd]) * sum_j softmax_j(scale q . k_j - slopes[hd] (i - j)) v_j,  j <= i = position.
 * Scores, softmax weights and sums are fp32 (the _bf16 prefill product carries every fp32 weight as three
 * bfloat16 terms).  q / caches as written by ohara_qkv_norm_append; gate (leading dimension ldg, in the
 * activation type; NULL: none); out rows of h*dv with leading dimension ldo, columns past h*dv are set to
 * zero up to the next multiple of 8 (ldo may go further).  dh, dv <= 256.  n_split > 1 (seq_len 1): the context of a (sequence, KV head) is cut into that many chunks
 * that meet in `workspace` (ohara_attn_bias_workspace_bytes, zero-filled once; calls sharing it must not
 * overlap). */
int64_t ohara_attn_bias_workspace_bytes(int rows, int h, int dv, int n_split);
int ohara_attn_bias_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int h, int h_kv, int dh,
                         int dv, int t_max, float scale, const float* slopes, const uint16_t* gate, int ldg, int n_split,
                         void* workspace, uint16_t* out, int ldo, const OharaSeq* seq, void* stream);
int ohara_attn_bias_f32(const float* q, const float* kcache, const float* vcache, int h, int h_kv, int dh, int dv,
                        int t_max, float scale, const float* slopes, const float* gate, int ldg, int n_split,
                        void* workspace, float* out, int ldo, const OharaSeq* seq, void* stream);

/* The same with other score functions and windows.  Score of query position i and key position j <= i:
 *   s = scale q . k_j;  cap > 0: s = cap tanh(s / cap);  slopes: s -= slopes[head] (i - j);
 * chunk > 0: only keys of the query's own chunk, floor(i / chunk) = floor(j / chunk), are visible.
 * ld_k, ld_v > 0: elements between neighbouring positions of the keys / values (0: h_kv * dhp, h_kv * dvp).
 * gate_elements: the gate has one entry per output element (rows of h*dv) instead of one per head.
 * window > 0: only the window keys up to and including the query's own are visible (with chunk: those of them in the chunk).
 * sinks: per head a score that joins the softmax without a value, p_j = exp(s_j) / (exp(sinks[head]) + sum exp(s)).
 * out_scale: factor of the output, applied before it is rounded.
 * d_shared > 0 (a multiple of 8): the last d_shared elements of every key, of all heads, are the d_shared elements of k_shared at its
 * position (positions ld_shared elements apart, rows as the keys'); the key rows then hold h_kv heads of dhp - d_shared elements.
 * ld_q > 0: elements between neighbouring rows of q (0: h * dhp). */
typedef struct OharaScores {
  float scale, cap;
  int chunk, gate_elements, ld_k, ld_v;
  const float* slopes;
  const float* sinks;
  int window;
  float out_scale;
  const void* k_shared;
  int ld_shared, d_shared, ld_q, reserved;
} OharaScores;
int ohara_attn_scored_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int h, int h_kv, int dh,
                           int dv, int t_max, const OharaScores* sc, const uint16_t* gate, int ldg, int n_split,
                           void* workspace, uint16_t* out, int ldo, const OharaSeq* seq, void* stream);
int ohara_attn_scored_f32(const float* q, const float* kcache, const float* vcache, int h, int h_kv, int dh, int dv,
                          int t_max, const OharaScores* sc, const float* gate, int ldg, int n_split, void* workspace,
                          float* out, int ldo, const OharaSeq* seq, void* stream);

/* Attention over the cache whose softmax weights are mixed across heads before they meet the values:
 *   w_h(i, j) = softmax_j(scale temp[h] q_h . k_j),  out_h(i) = sum_j (sum_g talk[h*H + g] w_g(i, j)) v_j,
 * H query heads on h_kv key/value heads, over j <= i with i - j < window (0: no window) or j < keep.  temp NULL: 1.  q (rows, h * dhp),
 * caches (cache rows, t_max, h_kv, dhp / dvp) with dhp, dvp = dh, dv rounded up to 8; out rows of ldo >= h * dv, zeros up to the next
 * multiple of 8.  dh, dv <= 256, h <= 256.  positions: no sequence ends past it.  One token per sequence: n_split chunks of the
 * visible positions, and the workspace starts zeroed once (it is left ready for the next call).  bf16 calls of 16 and more tokens per
 * sequence run on matrix products for up to 32 heads (16 with dh or dv over 128).  elem: bytes of an activation. */
typedef struct OharaMixedScores {
  float scale;
  int window, keep, reserved;
  const float* temp;
  const float* talk;
} OharaMixedScores;
int64_t ohara_attn_mixed_workspace_bytes(int batch, int seq_len, int h, int h_kv, int dh, int dv, int positions, int window, int keep,
                                         int n_split, int elem);
int ohara_attn_mixed_bf16(const uint16_t* q, const uint16_t* kcache, const uint16_t* vcache, int h, int h_kv, int dh, int dv, int t_max,
                          const OharaMixedScores* sc, int positions, int n_split, void* workspace, int64_t workspace_bytes, uint16_t* out,
                          int ldo, const OharaSeq* seq, void* stream);
int ohara_attn_mixed_f32(const float* q, const float* kcache, const float* vcache, int h, int h_kv, int dh, int dv, int t_max,
                         const OharaMixedScores* sc, int positions, int n_split, void* workspace, int64_t workspace_bytes, float* out,
                         int ldo, const OharaSeq* seq, void* stream);

/* Latent attention: all heads read one cached latent c (rank rp = rank rounded up to 8 per position) that is key and value at
 * once; a head's key and value projections are applied to its query and to its weighted sum instead.
 *   latent_front   p row [cq (q_rank) at 0; c (rank) at off_c]: each over its root mean square times qn / cn;
 *                  cq -> q_out (rows, q_rank rounded up to 8), c -> cache (cache rows, t_max, rp) and, if c_out, c_out (rows, rp)
 *   latent_rotary_front  p rows [h heads of dq unrotated and rp = rot rounded up to 8 rotated elements; the latent at off_c; the rotated
 *                  key part at off_r], rot (even) of the rotated elements in use: all rotated in neighbouring pairs by cos, sin
 *                  (positions, rot / 2) fp32; head i of the queries' part -> qr + row * ldqr + i * hqr (may be its place in p), the
 *                  latent over its root mean square times cn, followed by the key part -> cache (cache rows, t_max, rankp + rp)
 *                  and, if c_out, c_out (rows, rankp + rp).  cn NULL: queries only.  rank <= 512.
 *   head_linear    out[row, head, :] = W[head] x[row, head, :], W (h, n, k) row-major, n and k multiples of 8; x rows of ldx with
 *                  heads k apart; out rows of ldo with heads n_out <= n apart (entries n_out .. n-1 are dropped, columns past
 *                  h * n_out are set to zero);  gate (rows of ldg, h * n_out entries): times sigmoid(gate);
 *                  x_heads, out_heads > 0: elements between neighbouring heads of x / out (0: k / n_out; with out_heads > n_out
 *                  what lies between the heads is left alone)
 *   attn_latent    q (rows, h, rp) -> out (rows, h, rp): sum_j softmax_j(scale q . c_j) c_j over j <= position, rank <= 512.
 *                  d_key > 0 (a multiple of 8, <= 128): rows of q and of the cache end in d_key elements that take part in the
 *                  scores only.  window > 0: j > position - window
 *                  n_split > 1: the context is cut into that many chunks that meet in `workspace`
 *                  (ohara_attn_latent_workspace_bytes); a second launch merges them in chunk order. */
int ohara_latent_front_bf16(const uint16_t* p, int ldp, int q_rank, int off_c, int rank, const float* qn, const float* cn,
                            float eps, uint16_t* q_out, uint16_t* cache, int t_max, uint16_t* c_out, const OharaSeq* seq,
                            void* stream);
int ohara_latent_front_f32(const float* p, int ldp, int q_rank, int off_c, int rank, const float* qn, const float* cn,
                           float eps, float* q_out, float* cache, int t_max, float* c_out, const OharaSeq* seq,
                           void* stream);
int ohara_latent_rotary_front_bf16(uint16_t* p, int ldp, int h, int dq, int rot, const float* cos, const float* sin, uint16_t* qr, int ldqr,
                                   int hqr, int off_c, int off_r, int rank, const float* cn, float eps, uint16_t* cache, int t_max,
                                   uint16_t* c_out, const OharaSeq* seq, void* stream);
int ohara_latent_rotary_front_f32(float* p, int ldp, int h, int dq, int rot, const float* cos, const float* sin, float* qr, int ldqr, int hqr,
                                  int off_c, int off_r, int rank, const float* cn, float eps, float* cache, int t_max, float* c_out,
                                  const OharaSeq* seq, void* stream);
int ohara_head_linear_bf16(const uint16_t* x, int ldx, const uint16_t* w, int h, int n, int k, int n_out, int rows,
                           const uint16_t* gate, int ldg, uint16_t* out, int ldo, int x_heads, int out_heads, void* stream);
int ohara_head_linear_f32(const float* x, int ldx, const float* w, int h, int n, int k, int n_out, int rows, const float* gate,
                          int ldg, float* out, int ldo, int x_heads, int out_heads, void* stream);
int64_t ohara_attn_latent_workspace_bytes(int rows, int h, int rank, int n_split);
int ohara_attn_latent_bf16(const uint16_t* q, const uint16_t* cache, int h, int rank, int d_key, int t_max, float scale, int window, int n_split,
                           void* workspace, uint16_t* out, const OharaSeq* seq, void* stream);
int ohara_attn_latent_f32(const float* q, const float* cache, int h, int rank, int d_key, int t_max, float scale, int window, int n_split,
                          void* workspace, float* out, const OharaSeq* seq, void* stream);

/* Gated delta rule with one decay per head and key channel.  Per value head: S (dim x vdim) fp32,
 *   S <- diag(exp(lg)) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q,
 *   q, k, v: short causal convolution per channel (taps), silu; q, k over sqrt(sum of squares + 1e-6), q also times
 *   dim^-1/2;  lg = neg_a[head] * softplus(W_a2 a1 + dt_bias);  beta = sigmoid(b);
 *   out = o / rms(o) * norm_w * sigmoid(W_g2 g1).
 * A projection row p holds [q (kv_heads*dim); k (kv_heads*dim); v (heads*vdim)] from column 0, the rank_a columns a1
 * from off_a, the rank_g columns g1 from off_g (offsets and ranks multiples of 8) and the heads columns b from off_b.
 * a2 (heads*dim, rank_a), g2 (heads*vdim, rank_g) row-major in the activation type; conv_w (taps, channels) fp32 with the
 * current token's row last; state (cache rows, heads, dim, vdim rounded up to a multiple of 4) fp32; ring (cache rows,
 * taps, channels) in the activation type.  A sequence whose first token sits at position 0 starts from zero
 * whatever its state and ring hold.  dim, vdim <= 256.
 * a2 == NULL: one decay per head, lg = neg_a[head] * softplus(a + dt_bias[head]) with the heads columns a from off_a (any offset;
 * rank_a is not read).  g2 == NULL: the gate's heads*vdim columns come from off_g as they are (rank_g is not read).
 * flags: OHARA_DELTA_SILU_GATE: the gate is silu instead of sigmoid. */
#define OHARA_DELTA_SILU_GATE 1
typedef struct OharaDelta {
  int heads, kv_heads, dim, vdim, taps, rank_a, rank_g, off_a, off_g, off_b;
  float eps;
  int flags;
  const float* conv_w;
  const void* a2;
  const void* g2;
  const float* neg_a;
  const float* dt_bias;
  const float* norm_w;
} OharaDelta;
/* One token per sequence (seq_len 1): everything above in one launch; ring and state are updated. */
int ohara_delta_step_bf16(const OharaDelta* d, const uint16_t* p, int ldp, float* state, uint16_t* ring, uint16_t* out,
                          int ldo, const OharaSeq* seq, void* stream);
int ohara_delta_step_f32(const OharaDelta* d, const float* p, int ldp, float* state, float* ring, float* out, int ldo,
                         const OharaSeq* seq, void* stream);
/* Any number of tokens per sequence, in chunks of 32 tokens: za (rows, heads*dim) = W_a2 a1 and zg (rows, heads*vdim)
 * = W_g2 g1 come from the caller (NULL where a2 / g2 is).  First the chunks are solved on their own in parallel, then the state walks
 * over them on fp32 matrix products; state is updated, the ring is only read (follow with
 * ohara_conv_ring_store over the first 2*kv_heads*dim + heads*vdim columns of p).  workspace:
 * ohara_delta_workspace_bytes for the number of tokens per sequence worked on at a time (the call cuts
 * longer sequences into segments that fit); o_tmp: (rows, heads*vdim) fp32. */
int64_t ohara_delta_workspace_bytes(int heads, int dim, int vdim, int batch, int tokens);
int ohara_delta_prefill_bf16(const OharaDelta* d, const uint16_t* p, int ldp, const uint16_t* za, int ldza,
                             const uint16_t* zg, int ldzg, float* state, const uint16_t* ring, void* workspace,
                             int64_t workspace_bytes, float* o_tmp, uint16_t* out, int ldo, const OharaSeq* seq,
                             void* stream);
int ohara_delta_prefill_f32(const OharaDelta* d, const float* p, int ldp, const float* za, int ldza, const float* zg,
                            int ldzg, float* state, const float* ring, void* workspace, int64_t workspace_bytes,
                            float* o_tmp, float* out, int ldo, const OharaSeq* seq, void* stream);

/* Retention: linear attention with one fixed decay per head and no normaliser.  Per head, S (dim x vdim) fp32 from zero:
 *   S <- decay S + k_scale k v^T;   o = S^T q;   out = out_scale * o / sqrt(mean of o^2 over vdim_used + eps) * silu(g).
 * A projection row p holds q, k (heads*dim each), v, g (heads*vdim each) from columns off_q, off_k, off_v, off_g; dim, vdim and the
 * offsets are multiples of 8, vdim, dim <= 256; of each head's vdim columns the first vdim_used count (the others must be zero).
 * powers (heads, OHARA_RETENTION_CHUNK + 1) fp32: decay to the power of 0, 1, ...  state (cache rows, heads, dim, vdim) fp32; a
 * sequence whose first token sits at position 0 starts from zero whatever its state holds.  out: heads*vdim columns. */
#define OHARA_RETENTION_CHUNK 128
typedef struct OharaRetention {
  int heads, dim, vdim, vdim_used, off_q, off_k, off_v, off_g;
  float eps, k_scale, out_scale;
  int reserved;
  const float* powers;
} OharaRetention;
/* One token per sequence (seq_len 1), one launch. */
int ohara_retention_step_bf16(const OharaRetention* r, const uint16_t* p, int ldp, float* state, uint16_t* out, int ldo,
                              const OharaSeq* seq, void* stream);
int ohara_retention_step_f32(const OharaRetention* r, const float* p, int ldp, float* state, float* out, int ldo,
                             const OharaSeq* seq, void* stream);
/* Any number of tokens per sequence in chunks: what every chunk adds to the state (all chunks in parallel), the states before
 * the chunks, the outputs (in parallel again).  workspace: ohara_retention_workspace_bytes for the number of tokens per sequence
 * worked on at a time (the call cuts longer sequences into segments that fit). */
int64_t ohara_retention_workspace_bytes(int heads, int dim, int vdim, int batch, int tokens);
int ohara_retention_prefill_bf16(const OharaRetention* r, const uint16_t* p, int ldp, float* state, void* workspace,
                                 int64_t workspace_bytes, uint16_t* out, int ldo, const OharaSeq* seq, void* stream);
int ohara_retention_prefill_f32(const OharaRetention* r, const float* p, int ldp, float* state, void* workspace,
                                int64_t workspace_bytes, float* out, int ldo, const OharaSeq* seq, void* stream);

/* ---- routed experts with clamped gated units, fp32 router, groups, identity outputs ---------------------------------
 * router: z = W x in fp32 (w (n_out, k) row-major in the activation type), s = softmax(z) over all n_out outputs; the choice looks
 * at s + correction (fp32, NULL: s) inside the `keep` of `groups` equal groups of neighbouring outputs whose largest entry is
 * largest; the `top` best are chosen (ties: lowest index) -> idx (rows, top), weights s / (sum of the chosen s + 1e-20) -> wgt
 * (rows, top) fp32.  Sorted by expert: offs (n_out + 1), pair_of (rows*top) sorted position -> row*top + j, pos_of its inverse.
 * hist: workspace of ceil(rows*top / 1024) * n_out ints; counter: one zeroed int (left zero).  n_out <= 1024, top <= 64,
 * groups <= 64.  flags: OHARA_ROUTER_SIGMOID: s = sigmoid(z) instead (without a correction the choice follows z itself);
 * OHARA_ROUTER_PLAIN: the weights are the chosen s as they are. */
#define OHARA_ROUTER_SIGMOID 1
#define OHARA_ROUTER_PLAIN 2
int ohara_moe_router_bf16(const uint16_t* x, int ldx, const uint16_t* w, int ldw, const float* correction, int rows, int k, int n_out,
                          int top, int groups, int keep, int flags, int32_t* idx, float* wgt, int32_t* offs, int32_t* pair_of,
                          int32_t* pos_of, int32_t* hist, int32_t* counter, void* stream);
int ohara_moe_router_f32(const float* x, int ldx, const float* w, int ldw, const float* correction, int rows, int k, int n_out,
                         int top, int groups, int keep, int flags, int32_t* idx, float* wgt, int32_t* offs, int32_t* pair_of,
                         int32_t* pos_of, int32_t* hist, int32_t* counter, void* stream);
/* Products of the first n_experts experts over their sorted pairs.  glu: act[position] = clamped unit (ohara_gemm_glu_*) of row
 * pair_of[position] / top of x, with pair_w (NULL: none) of that row times pair_w[pair_of[position]]; down: y[position] = W_down act[position], not weighted.  bf16: packed weights expert_stride_bytes
 * apart; few pairs stream the weights (the shared expert, if given, rides along with its n_tokens rows), many run in tiles
 * of 128 (no shared expert).  f32: row-major (n_experts, n, k) matrices. */
int ohara_moe_glu_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int64_t expert_stride_bytes, int n_experts, int hidden, int d,
                       int top, int n_pairs, const int32_t* offs, const int32_t* pair_of, const float* pair_w, const OharaGlu* glu, uint16_t* act,
                       int ld_act, const uint16_t* wp_shared, int hidden_shared, int n_tokens, const OharaGlu* glu_shared,
                       uint16_t* act_shared, int ld_act_shared, void* stream);
int ohara_moe_down_bf16(const uint16_t* act, int ld_act, const uint16_t* wp, int64_t expert_stride_bytes, int n_experts, int d,
                        int hidden, int n_pairs, const int32_t* offs, uint16_t* y, int ldy, const uint16_t* wp_shared,
                        int hidden_shared, int n_tokens, const uint16_t* act_shared, int ld_act_shared, uint16_t* y_shared,
                        int ldy_shared, void* stream);
int ohara_moe_glu_f32(const float* x, int ldx, const float* w_gate, const float* w_up, int n_experts, int hidden, int d, int top,
                      int n_pairs, const int32_t* offs, const int32_t* pair_of, const float* pair_w, const OharaGlu* glu, float* act, int ld_act,
                      void* stream);
int ohara_moe_down_f32(const float* act, int ld_act, const float* w, int n_experts, int d, int hidden, int n_pairs,
                       const int32_t* offs, float* y, int ldy, void* stream);

/* ---- timing helpers (measurement only; no counterpart in the reference) -----------
 * Thin wrappers over hipEventCreate / hipEventDestroy / hipEventElapsedTime so that a
 * benchmark can time single launches on the stream they run on without another HIP
 * binding.  elapsed needs both events completed (synchronise the stream first). */
int ohara_event_create(void** event);
int ohara_event_destroy(void* event);
int ohara_event_record(void* event, void* stream);
int ohara_event_elapsed_ms(void* start, void* stop, float* ms);

#ifdef __cplusplus
}
#endif
#endif /* OHARA_DECODE_H */
