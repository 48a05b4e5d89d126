// Small memory-bound kernels of the decode step: embedding gather, standalone
// RMSNorm, greedy token selection and the device-side step bookkeeping.
#include "common.h"

namespace {

// out[t, :] = table[ids[t], :]   (nn.Embedding, ohara/models/llama.py:245,310)
__global__ __launch_bounds__(256) void embed_kernel(const int64_t* ids, const bf16_t* table, bf16_t* out, int d,
                                                    int vocab) {
  const int t = blockIdx.x;
  int64_t id = ids[t];
  if (id < 0 || id >= vocab) id = 0;  // the host validates ids; never read out of bounds
  const bf16_t* src = table + (size_t)id * d;
  bf16_t* dst = out + (size_t)t * d;
  if ((d & 7) == 0) {
    for (int i = threadIdx.x; i < d / 8; i += blockDim.x)
      reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
  } else {
    for (int i = threadIdx.x; i < d; i += blockDim.x) dst[i] = src[i];
  }
}

// ohara/modules/norm.py:16-21, one wave per row, which it holds in registers: read once, 16 bytes a lane, all loads in
// flight together (NC of them, for up to 512 NC columns).  A lane's eight columns and those of the lane 32 further are exchanged so that
// the squares are added column 256 after column 256, and the sums in the order of the kernel below: the same bits.
// Memory bound: 8192 x 768 takes 6.8 us, 4001 x 2048 6.9 (one workgroup per row, two bytes a lane, read twice: 9.9 and 10.6); 128 x
// 768, where it is the latency of one row, 2.1 (2.3).
template <int NC>
__global__ __launch_bounds__(256) void rmsnorm_wave_kernel(const bf16_t* x, const bf16_t* w, bf16_t* out, int rows, int d, float eps) {
  const int lane = threadIdx.x & 63;
  const size_t r = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (r >= (size_t)rows) return;
  uint4 v[NC], wv[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = 512 * c + 8 * lane;
    v[c] = i < d ? ldg16(x + r * d + i) : make_uint4(0, 0, 0, 0);
    wv[c] = i < d ? ldg16(w + i) : make_uint4(0, 0, 0, 0);
  }
  float s[4] = {0.f, 0.f, 0.f, 0.f};  // of columns 8 (lane & 31) + 4 (lane >> 5) + 0 .. 3, mod 256
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const u32x2 a = __builtin_amdgcn_permlane32_swap(v[c].x, v[c].z, false, false);
    const u32x2 b = __builtin_amdgcn_permlane32_swap(v[c].y, v[c].w, false, false);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[0] = __builtin_fmaf(lo_bf(a[h]), lo_bf(a[h]), s[0]);
      s[1] = __builtin_fmaf(hi_bf(a[h]), hi_bf(a[h]), s[1]);
      s[2] = __builtin_fmaf(lo_bf(b[h]), lo_bf(b[h]), s[2]);
      s[3] = __builtin_fmaf(hi_bf(b[h]), hi_bf(b[h]), s[3]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = lane_xor_sum<32>(lane_xor_sum<1>(lane_xor_sum<2>(lane_xor_sum<4>(s[e]))));
  const int q = __float_as_int((s[0] + s[2]) + (s[1] + s[3]));  // columns 64 (lane >> 3 & 3) .. + 63, mod 256
  const float tot = ((__int_as_float(__builtin_amdgcn_readlane(q, 0)) + __int_as_float(__builtin_amdgcn_readlane(q, 8))) +
                     __int_as_float(__builtin_amdgcn_readlane(q, 16))) + __int_as_float(__builtin_amdgcn_readlane(q, 24));
  const float rinv = 1.0f / sqrtf(tot / (float)d + eps);
  auto two = [&](uint32_t xx, uint32_t ww) {
    return pack_bf(rbf(lo_bf(xx) * rinv) * lo_bf(ww), rbf(hi_bf(xx) * rinv) * hi_bf(ww));
  };
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = 512 * c + 8 * lane;
    if (i < d)
      *reinterpret_cast<uint4*>(out + r * d + i) =
          make_uint4(two(v[c].x, wv[c].x), two(v[c].y, wv[c].y), two(v[c].z, wv[c].z), two(v[c].w, wv[c].w));
  }
}

// One workgroup per row: rows of any length and start.
__global__ __launch_bounds__(256) void rmsnorm_kernel(const bf16_t* x, const bf16_t* w, bf16_t* out, int d,
                                                      float eps) {
  const size_t r = blockIdx.x;
  const bf16_t* xr = x + r * d;
  __shared__ float red[4];
  float s = 0.f;
  for (int i = threadIdx.x; i < d; i += 256) {
    const float v = bf2f(xr[i]);
    s += v * v;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  const float tot = ((red[0] + red[1]) + red[2]) + red[3];
  const float rinv = 1.0f / sqrtf(tot / (float)d + eps);
  for (int i = threadIdx.x; i < d; i += 256) out[r * d + i] = f2bf(rbf(bf2f(xr[i]) * rinv) * bf2f(w[i]));
}

struct StepState {  // device-resident bookkeeping of a decode loop
  int32_t pos;      // cache position of the token being fed
  int32_t step;     // index of the token being produced
  int32_t done;     // workgroups of the selection kernel that have finished
  int32_t pad;
};

// Greedy selection: first index of the row maximum over the valid vocabulary
// (argmax of the last position, ohara/chat_engine.py:61-63, ohara/inference.py:40-45;
// padded ids masked as in chat_engine.py:398-399).  One workgroup per row.
// Writes next_ids[b] (fed back to the embedding) and, when `history` is given,
// history[step * B + b].  The last workgroup to finish advances pos and step.
__global__ __launch_bounds__(1024) void argmax_kernel(const bf16_t* logits, int ldl, int vocab, int valid,
                                                      int64_t* next_ids, int64_t* history, int hist_cap,
                                                      StepState* st, int B) {
  const int b = blockIdx.x;
  const bf16_t* row = logits + (size_t)b * ldl;
  const int n = min(valid, vocab);
  float best = -INFINITY;
  int bi = 0x7fffffff;
  auto take = [&](float v, int i) {
    if (v > best || (v == best && i < bi)) {
      best = v;
      bi = i;
    }
  };
  const int step = st && threadIdx.x == 0 ? st->step : 0;  // (before this workgroup counts itself out: nobody has moved it on)
  bool known = false;
  const bool wide = (ldl & 7) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0;
  const int n8 = wide ? n >> 3 : 0, wave = threadIdx.x >> 6;
  __shared__ float sv[16];
  __shared__ int si[16], first;
  if (n8 > 0) {
    // One CU walks the row, so the instructions of an id count: a thread's largest value and the place of it only where it is the row's.  Of
    // the patterns as 16-bit integers the largest signed one is the largest value if any is not negative, else the smallest unsigned one is:
    // an instruction an id; `key` orders what they give.  A NaN shows as a key above infinity's (or no number's at all): the row is walked
    // value by value then.  Eight loads of 16 bytes in flight a thread.  (A comparison of value and place for every id, four loads in
    // flight: from a graph 32 rows of 65536 ids 10.0 us, now 4.9; one of 32000 6.8, now 4.3.)
    typedef short s16x2 __attribute__((ext_vector_type(2)));
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    s16x2 hi = {-32768, -32768};
    u16x2 lo = {0xffff, 0xffff};
    uint4 v[8];
    for (int c0 = threadIdx.x; c0 < n8; c0 += 8 * 1024) {
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = ldg16(row + (size_t)min(c0 + u * 1024, n8 - 1) * 8);  // (past the end: the last eight once more)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          hi = __builtin_elementwise_max(hi, __builtin_bit_cast(s16x2, w[j]));
          lo = __builtin_elementwise_min(lo, __builtin_bit_cast(u16x2, w[j]));
        }
      }
    }
    int top = max((int)hi[0], (int)hi[1]);
    const int low = min((int)lo[0], (int)lo[1]);
    const int i_tail = (n8 << 3) + threadIdx.x;
    auto key_of = [](int bits) { return bits & 0x8000 ? 0x7fff - (bits & 0x7fff) : 0x8000 + bits; };
    int key = top >= 0 ? 0x8000 + top : 0x7fff - (low & 0x7fff);
    const int tail_key = i_tail < n ? key_of(row[i_tail]) : -1;
    if (threadIdx.x >= n8) key = -1;
    const int mine = max(key, tail_key);
    const int wtop = lanes_max<32, 1>(mine);
    if ((threadIdx.x & 63) == 0) si[wave] = wtop;
    if (threadIdx.x == 0) first = 0x7fffffff;
    __syncthreads();
    int m = si[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) m = max(m, si[i]);
    if (m <= 0x8000 + 0x7f80 && m >= 0x7fff - 0x7f80) {
      const float value = bf2f((bf16_t)(m & 0x8000 ? m & 0x7fff : 0x8000 | (0x7fff - m)));
      if (mine == m || (m == 0x8000 && mine == 0x7fff)) {  // (both zeros are the same value)
        int at = 0x7fffffff;
        if (threadIdx.x >= n8) {  // only the tail's value
        } else if (n8 <= 8 * 1024) {
#pragma unroll
          for (int u = 7; u >= 0; --u) {
            const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
            const int c = min((int)threadIdx.x + u * 1024, n8 - 1) * 8;
#pragma unroll
            for (int j = 3; j >= 0; --j) {
              if (hi_bf(w[j]) == value) at = c + 2 * j + 1;
              if (lo_bf(w[j]) == value) at = c + 2 * j;
            }
          }
        } else {
          for (int c = threadIdx.x; c < n8 && at == 0x7fffffff; c += 1024)
            for (int j = 7; j >= 0; --j)
              if (bf2f(row[8 * c + j]) == value) at = 8 * c + j;
        }
        if (i_tail < n && bf2f(row[i_tail]) == value) at = min(at, i_tail);
        atomicMin(&first, at);
      }
      __syncthreads();
      bi = first;
      known = true;
    }
  }
  if (!known) {
    for (int i = threadIdx.x; i < n; i += 1024) take(bf2f(row[i]), i);
    // NaN-free comparison network; ties resolve to the lowest index
    lane_xor_argmax<32>(best, bi);
    lane_xor_argmax<16>(best, bi);
    lane_xor_argmax<8>(best, bi);
    lane_xor_argmax<4>(best, bi);
    lane_xor_argmax<2>(best, bi);
    lane_xor_argmax<1>(best, bi);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
      sv[wave] = best;
      si[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 1; w < 16; ++w)
        if (sv[w] > best || (sv[w] == best && si[w] < bi)) {
          best = sv[w];
          bi = si[w];
        }
  }
  if (threadIdx.x == 0) {
    if (bi == 0x7fffffff) bi = 0;  // all -inf / NaN row
    next_ids[b] = bi;
    if (st) {
      if (history && step < hist_cap) history[(size_t)step * B + b] = bi;
      // only the counter is shared between workgroups: no fence, the ids are read by later kernels
      const int old = __hip_atomic_fetch_add(&st->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old == B - 1) {
        st->done = 0;
        st->pos += 1;
        st->step = step + 1;
      }
    }
  }
}

}  // namespace

namespace {
__global__ void advance_positions_kernel(int32_t* seq_pos, const uint8_t* active, int batch, int by) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < batch && (!active || active[b])) seq_pos[b] += by;
}
// the same, and the ids the next step feeds: what the step selected for an active sequence, 0 for an idle slot
__global__ void advance_ragged_kernel(int32_t* seq_pos, const uint8_t* active, const int64_t* new_ids, int64_t* next_ids,
                                      int batch, int by) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  const bool on = !active || active[b];
  if (on) seq_pos[b] += by;
  next_ids[b] = on ? new_ids[b] : 0;
}
// Slots that are taken or left; the host's numbers travel with the launch (a copy of each was a wait for the stream: 16 us, 48 of them
// for 16 sequences that leave, 32 behind the prompts of 16 that join; 16 prompts with 15 steps 10.7 -> 9.7 ms).
constexpr int SLOTS = 128;  // of a launch
struct Slots {
  int32_t slot[SLOTS], pos[SLOTS];
};
__global__ void set_slots_kernel(Slots s, int n, int active, const int64_t* ids, int64_t* next_ids, int32_t* seq_pos, uint8_t* flags) {
  const int i = threadIdx.x;
  if (i >= n) return;
  const int b = s.slot[i];
  seq_pos[b] = s.pos[i];
  flags[b] = (uint8_t)active;
  if (ids || !active) next_ids[b] = ids ? ids[i] : 0;
}
}  // namespace

extern "C" {

int ohara_abi_version(void) { return 1; }

int ohara_embed_bf16(const int64_t* ids, const uint16_t* table, uint16_t* out, int n_tokens, int d, int vocab,
                     void* stream) {
  if (!ids || !table || !out || n_tokens < 1 || d < 1 || vocab < 1) return OHARA_EINVAL;
  hipLaunchKernelGGL(embed_kernel, dim3(n_tokens), dim3(256), 0, (hipStream_t)stream, ids, table, out, d, vocab);
  return ohara_launch_status();
}

int ohara_rmsnorm_bf16(const uint16_t* x, const uint16_t* w, uint16_t* out, int rows, int d, float eps,
                       void* stream) {
  if (!x || !w || !out || rows < 1 || d < 1) return OHARA_EINVAL;
  if ((d & 7) == 0 && d <= 4096 && (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0) {
    const int waves = rows < 1024 ? 1 : 4;  // few rows: over as many CUs as there are
    auto kernel = d <= 512 ? rmsnorm_wave_kernel<1> : d <= 1024 ? rmsnorm_wave_kernel<2> : d <= 2048 ? rmsnorm_wave_kernel<4>
                                                                                                     : rmsnorm_wave_kernel<8>;
    hipLaunchKernelGGL(kernel, dim3((rows + waves - 1) / waves), dim3(64 * waves), 0, (hipStream_t)stream, x, w, out, rows, d, eps);
    return ohara_launch_status();
  }
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(256), 0, (hipStream_t)stream, x, w, out, d, eps);
  return ohara_launch_status();
}

int ohara_argmax_bf16(const uint16_t* logits, int ldl, int batch, int vocab, int valid_vocab, int64_t* next_ids,
                      int64_t* history, int hist_cap, int32_t* step_state, void* stream) {
  if (!logits || !next_ids || batch < 1 || vocab < 1 || valid_vocab < 1 || ldl < vocab) return OHARA_EINVAL;
  hipLaunchKernelGGL(argmax_kernel, dim3(batch), dim3(1024), 0, (hipStream_t)stream, logits, ldl, vocab,
                     valid_vocab, next_ids, history, hist_cap, reinterpret_cast<StepState*>(step_state), batch);
  return ohara_launch_status();
}

}  // extern "C"

extern "C" int ohara_advance_positions(int32_t* seq_pos, const uint8_t* active, int batch, int by, void* stream) {
  if (!seq_pos || batch < 1) return OHARA_EINVAL;
  hipLaunchKernelGGL(advance_positions_kernel, dim3((batch + 255) / 256), dim3(256), 0, (hipStream_t)stream, seq_pos,
                     active, batch, by);
  return ohara_launch_status();
}

extern "C" int ohara_advance_ragged(int32_t* seq_pos, const uint8_t* active, const int64_t* new_ids, int64_t* next_ids,
                                    int batch, int by, void* stream) {
  if (!seq_pos || !new_ids || !next_ids || batch < 1) return OHARA_EINVAL;
  hipLaunchKernelGGL(advance_ragged_kernel, dim3((batch + 255) / 256), dim3(256), 0, (hipStream_t)stream, seq_pos,
                     active, new_ids, next_ids, batch, by);
  return ohara_launch_status();
}

extern "C" int ohara_set_slots(const int32_t* slots, const int32_t* positions, int n, int active, const int64_t* ids, int64_t* next_ids,
                               int32_t* seq_pos, uint8_t* active_flags, int batch, void* stream) {
  if (!slots || !next_ids || !seq_pos || !active_flags || n < 1 || batch < 1) return OHARA_EINVAL;
  for (int i = 0; i < n; ++i)
    if (slots[i] < 0 || slots[i] >= batch) return OHARA_EINVAL;
  for (int i0 = 0; i0 < n; i0 += SLOTS) {
    const int m = n - i0 < SLOTS ? n - i0 : SLOTS;
    Slots s{};
    for (int i = 0; i < m; ++i) {
      s.slot[i] = slots[i0 + i];
      s.pos[i] = positions ? positions[i0 + i] : 0;
    }
    hipLaunchKernelGGL(set_slots_kernel, dim3(1), dim3(SLOTS), 0, (hipStream_t)stream, s, m, active ? 1 : 0, ids ? ids + i0 : nullptr, next_ids,
                       seq_pos, active_flags);
  }
  return ohara_launch_status();
}
