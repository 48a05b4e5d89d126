#!/usr/bin/env python3
"""Decode benchmark of the MI355X KV-cache decode path.

One "step" = one decode step (one new token for every sequence of the batch) of the d12
Llama (d_model 768, 12 layers, 6 heads x 128, SwiGLU 3072, vocab 65536, bf16, random-init
N(0, 0.02) seed 0) after a 1024-token prompt, through the KV cache (capacity 4096).
Inputs (weights, prompt, cache) are resident in HBM before the timed region.

    python bench.py [--gpus 1] [--steps 256] [--warmup 16]

prints ONE JSON line: decode tokens/s at batch 1 (the configuration the >= 70 %-of-HBM
target is quoted on) with the same measurement at batch 8/32/64 under "also", the
roofline of the dominant kernel measured with HIP events inside real decode steps, and the
CPU oracle timed on this host's cores.
"""

from __future__ import annotations

import argparse
import ctypes as C
import json
import os
import sys
import time

import torch

HBM_PEAK_GBS = 8000.0

# HBM bytes per launch of the persistent decode kernel at batch 1, prompt 1024, from two
# rocprofv3 --pmc runs of this script (FETCH_SIZE, then WRITE_SIZE), each scaled by what the same
# counter reads for a 1 GiB copy (--pmc-calibration): 375.6 MB read + 1.3 MB written.  Counters
# cannot be read from inside this process, so the figure is carried here; the runs and the
# arithmetic are in profiles/decode_mega_kernel_d12_batch1_pmc.txt.
PMC_TRAFFIC_BYTES = {("persistent", 1, 1024): 377.2e6}

D12 = dict(vocab_size=65536, hidden_size=768, intermediate_size=3072, num_attention_heads=6,
           num_key_value_heads=0, num_hidden_layers=12, max_sequence_length=4096, dropout=0.0)


def d12_state(device, seed=0):
    """Random-init weights of the reference's shapes, N(0, 0.02), unit norm weights."""
    from ohara_amd.llama import Config

    cfg = Config(**D12)
    g = torch.Generator(device=device).manual_seed(seed)
    d, f, v = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size

    def n(*shape):
        return (torch.randn(*shape, generator=g, device=device) * 0.02).to(torch.bfloat16)

    st = {"token_emb.weight": n(v, d), "vocab_proj.weight": n(v, d),
          "norm.weight": torch.ones(d, dtype=torch.bfloat16, device=device)}
    for i in range(cfg.num_hidden_layers):
        p = f"layers.{i}."
        for nm in ("key", "query", "value", "proj"):
            st[p + f"attn.{nm}.weight"] = n(d, d)
        st[p + "ff.up.weight"] = n(f, d)
        st[p + "ff.gate.weight"] = n(f, d)
        st[p + "ff.down.weight"] = n(d, f)
        st[p + "norm1.weight"] = torch.ones(d, dtype=torch.bfloat16, device=device)
        st[p + "norm2.weight"] = torch.ones(d, dtype=torch.bfloat16, device=device)
    return cfg, st


def step_bytes(cfg, batch, length, int8=False):
    """Algorithmic HBM bytes of one decode step at cached length `length` (after append); int8: the caches hold one
    byte per value plus an fp32 (scale, minimum) pair per head row."""
    d, f, v, nl = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.num_hidden_layers
    params = nl * (4 * d * d + 3 * d * f) + v * d + (2 * nl + 1) * d
    kv_row = nl * 2 * d * 2
    if int8:
        kv_row = nl * 2 * (d + 8 * (cfg.num_key_value_heads or cfg.num_attention_heads))
    return 2 * params + batch * (kv_row * length + kv_row + 2 * d + 2 * v)


def lm_head_bytes(cfg, batch):
    d, v = cfg.hidden_size, cfg.vocab_size
    return 2 * (v * d + d) + batch * 2 * (d + v)


def time_decode(model, batch, prompt_len, warmup, steps, seed=0, persistent=None, sampling=None, int8=False):
    g = torch.Generator().manual_seed(seed)
    prompt = torch.randint(0, model.config.vocab_size, (batch, prompt_len), generator=g).to(model.device)
    u = None
    if sampling is not None:  # one fixed, seeded tensor of uniform draws for the whole run
        u = torch.rand(warmup + steps + 8, batch, generator=g).to(model.device)
    sess = model.session(batch, warmup + steps + 8, persistent=persistent, sampling=sampling, u=u,
                         kv_cache=model.build_kv_cache(batch, int8=True) if int8 else None)
    sess.prefill(prompt)
    sess.capture()
    sess.run(max(0, warmup - 1))
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    sess.run(steps)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    sess.check_error()
    l_mean = prompt_len + warmup + (steps + 1) / 2.0
    return dt, l_mean, sess


def time_kernel_in_situ(sess, kernel_index, steps):
    """Average duration of launch `kernel_index` inside real (eager) decode steps, from HIP
    events recorded on the launch stream right before and after that launch."""
    from ohara_amd._lib import check, lib

    L = lib()
    evs = []
    for _ in range(steps):
        a, b = C.c_void_p(), C.c_void_p()
        check(L.ohara_event_create(C.byref(a)), "event")
        check(L.ohara_event_create(C.byref(b)), "event")
        evs.append((a, b))
    for a, b in evs:
        sess.step(prof_kernel=kernel_index, prof_start=a, prof_stop=b)
    torch.cuda.synchronize()
    tot = 0.0
    for a, b in evs:
        ms = C.c_float()
        check(L.ohara_event_elapsed_ms(a, b, C.byref(ms)), "elapsed")
        tot += ms.value
        L.ohara_event_destroy(a)
        L.ohara_event_destroy(b)
    return tot / steps * 1e-3


def cpu_baseline(budget_s=20.0):
    """The CPU oracle (a PyTorch restatement of the reference's eager path) on this host:
    d12 Llama in fp32, batch 1, 128-token prompt, greedy decode through the KV cache."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    from oracle import llama_ref as R

    cores = torch.get_num_threads()
    rcfg = R.RefConfig(**D12)
    w = R.init_weights(rcfg, seed=0, dtype=torch.float32)
    ref = R.RefLlama(rcfg, w)
    prompt = torch.randint(0, rcfg.vocab_size, (1, 128), generator=torch.Generator().manual_seed(0))
    cache = ref.build_kv_cache(1)
    t0 = time.perf_counter()
    logits = ref(prompt, cache, 0)
    prefill_s = time.perf_counter() - t0
    nxt = logits[:, -1].argmax(-1, keepdim=True)
    pos, n = 128, 0
    for _ in range(4):  # warm-up
        nxt = ref(nxt, cache, pos)[:, -1].argmax(-1, keepdim=True)
        pos += 1
    t0 = time.perf_counter()
    while n < 512 and time.perf_counter() - t0 < budget_s:  # about 14 s on 16 cores
        nxt = ref(nxt, cache, pos)[:, -1].argmax(-1, keepdim=True)
        pos += 1
        n += 1
    dt = time.perf_counter() - t0
    return {
        "value": round(n / dt, 2), "unit": "tokens/s", "cores": cores, "kind": "port",
        "sample": f"d12 Llama fp32, batch 1, prompt 128 (prefill {prefill_s:.2f}s), {n} greedy decode steps "
                  f"through the KV cache, torch {torch.__version__} CPU, {os.cpu_count()} logical CPUs visible",
    }


# ---------------------------------------------------------------------------------------------
# Per-kernel figures of the other configurations (attention microbench, prefill on MFMA, BitNet
# ternary decode, MoE decode).  Each is timed as a HIP graph replay, so host launch cost is out.
# ---------------------------------------------------------------------------------------------
MFMA_BF16_PEAK_TFLOPS = 2500.0


def graph_time(fn, iters=10):
    """Seconds per call of fn(), captured once into a HIP graph and replayed `iters` times."""
    fn()
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(iters):
        g.replay()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / iters * 1e-3


def bench_attention_microbench(dev):
    """GQA decode attention, 32 query / 8 KV heads x 128, one query per sequence over L cached
    positions.  Algorithmic bytes: K + V (4*Hkv*D*B*L) + Q and O (4*H*D*B)."""
    from ohara_amd import ops
    from ohara_amd.llama import KVCache

    H, Hkv, D = 32, 8, 128
    out = []
    for B, L in ((b, l) for b in (1, 16, 64) for l in (1024, 4096, 16384, 32768)):
        ns = max(1, min(1024 // (B * Hkv), L // 128, 64))
        g = torch.Generator(device=dev).manual_seed(1)
        q = torch.randn(B, H * D, device=dev, generator=g).to(torch.bfloat16)
        k = torch.randn(B, L, Hkv, D, device=dev, generator=g).to(torch.bfloat16)
        v = torch.randn(B, L, Hkv, D, device=dev, generator=g).to(torch.bfloat16)
        ws = ops.attn_workspace(B, H, Hkv, D, ns, dev)
        o = torch.empty(B, H * D, device=dev, dtype=torch.bfloat16)
        t = graph_time(lambda: ops.attn_decode(q, k, v, H, Hkv, D, L, ns, ws, o))
        by = 4.0 * Hkv * D * B * L + 4.0 * H * D * B
        row = {"batch": B, "context": L, "n_split": ns, "us": round(t * 1e6, 1), "GBs": round(by / t / 1e9, 1),
               "frac_of_hbm_peak": round(by / t / 1e9 / HBM_PEAK_GBS, 4)}
        # the same rows through the int8 cache: codes (1 byte) + an fp32 scale and minimum per row
        cache = KVCache((B, L, Hkv, D), L, device=dev, dtype=torch.bfloat16, int8=True)
        step = max(1, 4096 // B)
        for p0 in range(0, L, step):
            ops.kv_quant_append(k[:, p0:p0 + step].contiguous(), v[:, p0:p0 + step].contiguous(), cache, p0)
        t8 = graph_time(lambda: ops.attn_cached_int8(q, cache, H, Hkv, D, L - 1, ns, ws, o))
        by8 = 2.0 * Hkv * (D + 8) * B * L + 4.0 * H * D * B
        row["int8_cache"] = {"us": round(t8 * 1e6, 1), "GBs": round(by8 / t8 / 1e9, 1),
                             "frac_of_hbm_peak": round(by8 / t8 / 1e9 / HBM_PEAK_GBS, 4)}
        out.append(row)
        del q, k, v, ws, o, cache
        torch.cuda.empty_cache()
    return out


def bench_continuous(model, cfg, dev, slots=32, steps=128):
    """Continuous batching: `slots` sequences of different lengths (prompts of 256..1279 tokens)
    decode in one batch, every slot at its own cache position; one graph replay per step."""
    from ohara_amd.batching import ContinuousBatcher

    g = torch.Generator().manual_seed(4)
    lens = torch.randint(256, 1280, (slots,), generator=g).tolist()
    bat = ContinuousBatcher(model, slots)
    for n in lens:
        bat.add(torch.randint(0, cfg.vocab_size, (n,), generator=g))
    for _ in range(8):
        bat.step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        bat.step()
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / steps
    mean_len = sum(lens) / slots + 8 + steps / 2
    by = step_bytes(cfg, slots, mean_len)
    return {"slots": slots, "prompt_lengths": "uniform 256..1279", "mean_context": round(mean_len, 1),
            "ms_per_step": round(dt * 1e3, 4), "tokens_per_s": round(slots / dt, 1),
            "frac_of_hbm_peak": round(by / dt / 1e9 / HBM_PEAK_GBS, 4),
            "note": "host reads the new ids every step (one synchronisation per step)"}


def bench_chat_engine(model, cfg, dev, prompt_len=1024, new_tokens=256, warmup=16):
    """The reference's caller-facing API on the same workload: ChatEngine.generate (render, prefill,
    device-resident sampled decode, stop check and incremental detokenisation on the host) with the
    reference's chat defaults (temperature 0.8, top-p 0.95, no top-k), against a bare decode session
    with the same sampler.  Tokens/s of the API leg count the whole call, prompt prefill included."""
    from ohara_amd.chat_engine import ChatEngine
    from ohara_amd.sampling import SamplingConfig

    class Tok:  # one printable character per id
        eos_token_id = None
        bos_token_id = None

        def __len__(self):
            return cfg.vocab_size

        def get_vocab(self):
            return {}

        def decode(self, ids, skip_special_tokens=True):
            return "".join(chr(0x4E00 + (i % 0x5000)) for i in ids)

    g = torch.Generator().manual_seed(9)
    prompt = torch.randint(0, cfg.vocab_size, (prompt_len,), generator=g).tolist()
    eng = ChatEngine(model, Tok(), renderer=lambda tok, turns, max_tokens: prompt, stop_ids=())
    sc = SamplingConfig(temperature=0.8, top_p=0.95, max_new_tokens=new_tokens)
    msgs = [{"role": "user", "content": "x"}]
    eng.generate(msgs, sc, seed=0)  # builds the session and captures the graph
    torch.cuda.synchronize()
    best = None
    for rep in range(3):
        t0 = time.perf_counter()
        text = eng.generate(msgs, sc, seed=1 + rep)
        dt = time.perf_counter() - t0
        assert len(text) == new_tokens
        best = dt if best is None else min(best, dt)
    dts, _, sess = time_decode(model, 1, prompt_len, warmup, new_tokens, sampling=sc)
    del sess
    api, bare = new_tokens / best, new_tokens / dts
    return {"tokens_per_s": round(api, 1), "ms_per_token": round(best / new_tokens * 1e3, 4),
            "new_tokens": new_tokens, "prompt_len": prompt_len,
            "sampling": "temperature 0.8, top-p 0.95 (ohara/chat_engine.py:35-37 defaults)",
            "bare_session_tokens_per_s": round(bare, 1), "api_over_session": round(api / bare, 3),
            "note": "ChatEngine.generate end to end (prefill of the prompt, chunked read-back, stop check, "
                    "whole-reply detokenisation per token); the session figure is decode steps only"}


def bench_prefill(model, cfg, dev):
    """Batched prefill of the d12 model (1024 tokens per sequence) and its MFMA kernels alone."""
    from ohara_amd import ops

    res = {}
    B, S = 8, 1024
    prompt = torch.randint(0, cfg.vocab_size, (B, S), device=dev)
    for _ in range(2):
        cache = model.build_kv_cache(B)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        model(prompt, cache, 0, last_only=True)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
    d, f = cfg.hidden_size, cfg.intermediate_size
    flops = 2.0 * B * S * cfg.num_hidden_layers * (4 * d * d + 3 * d * f) + 4.0 * B * d * S * (S + 1) / 2 * cfg.num_hidden_layers
    res["d12_prefill"] = {"batch": B, "prompt": S, "ms": round(dt * 1e3, 3), "tokens_per_s": round(B * S / dt, 1),
                          "TFLOPs": round(flops / dt / 1e12, 1)}
    del cache
    M = B * S
    x = torch.randn(M, f, device=dev).to(torch.bfloat16)
    kern = []
    for name, n, k, kind in (("qkv 2304x768", 3 * d, d, "store"), ("wo 768x768", d, d, "store"),
                             ("gate/up 2x3072x768 + SwiGLU", f, d, "swiglu"), ("down 768x3072", d, f, "store")):
        if kind == "swiglu":
            wp = ops.pack_gate_up((torch.randn(n, k, device=dev) * 0.02).to(torch.bfloat16),
                                  (torch.randn(n, k, device=dev) * 0.02).to(torch.bfloat16))
            fl = 2.0 * M * 2 * n * k
        else:
            wp = ops.pack_linear((torch.randn(n, k, device=dev) * 0.02).to(torch.bfloat16))
            fl = 2.0 * M * n * k
        o = torch.empty(M, n, device=dev, dtype=torch.bfloat16)
        xin = x[:, :k]
        t = graph_time(lambda: ops.gemm(xin, wp, out=o), iters=50)
        kern.append({"kernel": "gemm_tile_kernel " + name, "rows": M, "us": round(t * 1e6, 1),
                     "TFLOPs": round(fl / t / 1e12, 1), "mfma_util": round(fl / t / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4)})
    H, D = cfg.num_attention_heads, d // cfg.num_attention_heads
    q = torch.randn(M, d, device=dev).to(torch.bfloat16)
    kk = torch.randn(B, S, H, D, device=dev).to(torch.bfloat16)
    vv = torch.randn(B, S, H, D, device=dev).to(torch.bfloat16)
    o = torch.empty_like(q)
    t = graph_time(lambda: ops.attn_prefill(q, kk, vv, H, H, D, 0, S, o))
    fl = 4.0 * B * H * D * S * (S + 1) / 2
    kern.append({"kernel": "attn_prefill, heads of 128, causal", "rows": M, "us": round(t * 1e6, 1),
                 "TFLOPs": round(fl / t / 1e12, 1), "mfma_util": round(fl / t / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4)})
    res["mfma_kernels"] = kern
    return res


def _fill_cache(cache, length, batch):
    for c in cache:
        c.key.normal_()
        c.value.normal_()
        c.length, c.batch_size = length, batch


def bitnet_c4_state(dev, n_layers=24, t_max=2048):
    """Config and state dict of the BitNet-b1.58 ternary Llama (d 2048, 16 x 128 heads, FFN 5632,
    vocab 32000): ternary weights uniform over {-1, 0, 1} (seed 2) with a per-tensor scale, unit norms."""
    from ohara_amd.bitnet import BIT_TARGETS
    from ohara_amd.llama import Config

    cfg = Config(vocab_size=32000, hidden_size=2048, intermediate_size=5632, num_attention_heads=16,
                 num_key_value_heads=0, num_hidden_layers=n_layers, max_sequence_length=t_max, dropout=0.0)
    g = torch.Generator(device=dev).manual_seed(2)
    d, f, v = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size
    shapes = {"attn.key": (d, d), "attn.query": (d, d), "attn.value": (d, d), "attn.proj": (d, d),
              "ff.gate": (f, d), "ff.up": (f, d), "ff.down": (d, f)}
    st = {"token_emb.weight": (torch.randn(v, d, device=dev, generator=g) * 0.02).to(torch.bfloat16),
          "vocab_proj.weight": (torch.randn(v, d, device=dev, generator=g) * 0.02).to(torch.bfloat16),
          "norm.weight": torch.ones(d, device=dev, dtype=torch.bfloat16)}
    for i in range(cfg.num_hidden_layers):
        p = f"layers.{i}."
        for nm in BIT_TARGETS:
            n, k = shapes[nm]
            st[p + nm + ".ternary"] = torch.randint(-1, 2, (n, k), device=dev, generator=g, dtype=torch.int8)
            st[p + nm + ".gamma"] = torch.tensor(0.02)
            st[p + nm + ".rms_norm.weight"] = torch.ones(k, device=dev, dtype=torch.bfloat16)
        st[p + "norm1.weight"] = torch.ones(d, device=dev, dtype=torch.bfloat16)
        st[p + "norm2.weight"] = torch.ones(d, device=dev, dtype=torch.bfloat16)
    return cfg, st


def bench_bitnet(dev, batches=(1, 8)):
    """BitNet-b1.58 ternary Llama (d 2048, 24 layers, 16 x 128 heads, FFN 5632, vocab 32000):
    one decode step at context 2048, batch 1 and 8."""
    from ohara_amd.bitnet import BitLlama

    cfg, st = bitnet_c4_state(dev)
    d, v = cfg.hidden_size, cfg.vocab_size
    model = BitLlama(cfg, st, device=dev)
    del st
    out = []
    L = cfg.max_sequence_length
    for B in batches:
        cache = model.build_kv_cache(B)
        ids = torch.randint(0, v, (B, 1), device=dev)

        def step():
            _fill_len(cache, L - 1, B)
            return model(ids, cache, L - 1, last_only=True)

        _fill_cache(cache, L - 1, B)
        t = graph_time(step)
        by = model.packed_weight_bytes() + 2.0 * v * d + 2.0 * 2 * d * cfg.num_hidden_layers * B * L
        row = {"batch": B, "context": L, "launch": "chain of 5 kernels per layer", "ms_per_step": round(t * 1e3, 4),
               "tokens_per_s": round(B / t, 1), "step_bytes": int(by), "GBs": round(by / t / 1e9, 1),
               "frac_of_hbm_peak": round(by / t / 1e9 / HBM_PEAK_GBS, 4)}
        out.append(row)
        if model.supports_persistent(B):
            # the single-launch step on the same caches: every replay starts from position L - 1 again
            sess = model.session(B, 4, kv_cache=cache, persistent=True)
            _fill_len(cache, 0, B)
            sess.prefill(ids)
            _fill_cache(cache, L - 1, B)
            start = torch.tensor([L - 1, 1, 0, 0], dtype=torch.int32, device=dev)

            def pstep():
                sess.step_state.copy_(start)
                sess._launch_step()

            tp = graph_time(pstep)
            sess.check_error()
            out.append(dict(row, launch="one persistent kernel per step", ms_per_step=round(tp * 1e3, 4),
                            tokens_per_s=round(B / tp, 1), GBs=round(by / tp / 1e9, 1),
                            frac_of_hbm_peak=round(by / tp / 1e9 / HBM_PEAK_GBS, 4)))
            del sess
        del cache
        torch.cuda.empty_cache()
    return out


def _fill_len(cache, length, batch):
    for c in cache:
        c.length, c.batch_size = length, batch


def moe_c5_state(dev, n_layers=16, t_max=2048):
    """Config and state dict of the MoE Llama (d 1024, 16 x 64 heads, 64 routed SwiGLU experts of
    hidden 512, top-8, one shared expert, softmax router): bf16 N(0, 0.02) seed 3, router rows
    N(0, 1/d) so that the router logits spread like N(0, 1)."""
    from ohara_amd.llama import Config

    cfg = Config(vocab_size=32000, hidden_size=1024, intermediate_size=512, num_attention_heads=16,
                 num_key_value_heads=0, num_hidden_layers=n_layers, max_sequence_length=t_max, dropout=0.0,
                 moe_num_experts=64, moe_experts_per_tok=8, moe_grouped=True, moe_num_shared_experts=1)
    g = torch.Generator(device=dev).manual_seed(3)
    d, f, v, E = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.moe_num_experts

    def n(*shape):
        return (torch.randn(*shape, device=dev, generator=g) * 0.02).to(torch.bfloat16)

    one = lambda: torch.ones(d, device=dev, dtype=torch.bfloat16)  # noqa: E731
    st = {"token_emb.weight": n(v, d), "vocab_proj.weight": n(v, d), "norm.weight": one()}
    for i in range(cfg.num_hidden_layers):
        p = f"layers.{i}."
        for nm in ("key", "query", "value", "proj"):
            st[p + f"attn.{nm}.weight"] = n(d, d)
        st[p + "ff.w_gate"], st[p + "ff.w_up"], st[p + "ff.w_down"] = n(E, d, f), n(E, d, f), n(E, f, d)
        st[p + "ff.router.weight"] = (torch.randn(E, d, device=dev, generator=g) / d ** 0.5).to(torch.bfloat16)
        st[p + "ff.router_bias"] = torch.zeros(E, device=dev, dtype=torch.bfloat16)
        st[p + "ff.shared_gate.weight"], st[p + "ff.shared_up.weight"] = n(f, d), n(f, d)
        st[p + "ff.shared_down.weight"] = n(d, f)
        st[p + "norm1.weight"], st[p + "norm2.weight"] = one(), one()
    return cfg, st


def bench_moe(dev):
    """MoE decode (16 layers, d 1024, 16 x 64 heads, 64 routed SwiGLU experts of hidden 512, top-8,
    one shared expert): one step of 64 sequences at context 2048."""
    from ohara_amd.moe import MoeLlama

    cfg, st = moe_c5_state(dev)
    d, f, v, E = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.moe_num_experts
    model = MoeLlama(cfg, st, device=dev)
    del st
    B, L = 64, cfg.max_sequence_length
    cache = model.build_kv_cache(B)
    _fill_cache(cache, L - 1, B)
    ids = torch.randint(0, v, (B, 1), device=dev)

    def step():
        _fill_len(cache, L - 1, B)
        return model(ids, cache, L - 1, last_only=True)

    t = graph_time(step, iters=5)
    nl = cfg.num_hidden_layers
    expert_b = nl * 3.0 * E * d * f * 2
    by = expert_b + nl * (3.0 * d * f + 4.0 * d * d + E * d) * 2 + 2.0 * v * d + 2.0 * 2 * d * nl * B * L
    flops = nl * 2.0 * 3 * (B * cfg.moe_experts_per_tok) * d * f
    return {"batch": B, "context": L, "ms_per_step": round(t * 1e3, 4), "tokens_per_s": round(B / t, 1),
            "step_bytes": int(by), "GBs": round(by / t / 1e9, 1), "frac_of_hbm_peak": round(by / t / 1e9 / HBM_PEAK_GBS, 4),
            "expert_ffn_TFLOPs_if_all_time": round(flops / t / 1e12, 2),
            "bound": "hbm (about 8 rows per expert: ~8 flop/byte)"}


def phi2_model(dev):
    """Phi-2 shape (32 layers, d 2560, 32 x 80 heads, 32 rotated features, MLP 10240, vocab 51200)
    with random bf16 weights."""
    from ohara_amd.phi import Phi, PhiConfig

    cfg = PhiConfig()
    g = torch.Generator(device=dev).manual_seed(4)
    d, f, v = cfg.hidden_size, cfg.multiple_of * cfg.hidden_size, cfg.vocab_size

    def n(*shape):
        return (torch.randn(*shape, device=dev, generator=g) * 0.02).to(torch.bfloat16)

    st = {"wte.weight": n(v, d), "lm_head.weight": n(v, d), "lm_head.bias": n(v), "ln.weight": torch.ones(d, device=dev),
          "ln.bias": n(d)}
    for i in range(cfg.num_hidden_layers):
        p = f"layers.{i}."
        st[p + "ln.weight"], st[p + "ln.bias"] = torch.ones(d, device=dev), n(d)
        for nm in ("q_proj", "k_proj", "v_proj", "dense"):
            st[p + f"mixer.{nm}.weight"], st[p + f"mixer.{nm}.bias"] = n(d, d), n(d)
        st[p + "mlp.fc1.weight"], st[p + "mlp.fc1.bias"] = n(f, d), n(f)
        st[p + "mlp.fc2.weight"], st[p + "mlp.fc2.bias"] = n(d, f), n(d)
    model = Phi(cfg, st, device=dev)
    del st
    torch.cuda.empty_cache()
    return cfg, model


def phi_decode_only(dev, batch, steps=12, context=1024):
    """Eager Phi-2 decode steps over a randomly filled cache and nothing else: the workload of the
    per-kernel profiles (`--phi-decode-only B`)."""
    from ohara_amd import ops

    cfg, model = phi2_model(dev)
    cache = model.build_kv_cache(batch)
    for c in cache:
        c.key.normal_()
        c.value.normal_()
    ids = torch.randint(0, cfg.vocab_size, (batch,), device=dev)
    state = torch.tensor([context, 0, 0, 0], dtype=torch.int32, device=dev)
    for _ in range(steps):
        lg = model._run(ids, batch, 1, cache, 0, state, False)
        ops.argmax(lg, next_ids=ids, step_state=state)
    torch.cuda.synchronize()
    return {"batch": batch, "steps": steps, "context_end": int(state[0])}


def bench_phi(dev):
    """Phi-2 shape, random bf16 weights: greedy decode at batch 1 and 8 after a 1024-token context, one
    graph replay per step (5 launches per layer)."""
    cfg, model = phi2_model(dev)
    d, f, v = cfg.hidden_size, cfg.multiple_of * cfg.hidden_size, cfg.vocab_size
    nl, ctx, steps = cfg.num_hidden_layers, 1024, 64
    weight_b = 2.0 * (nl * (4 * d * d + 2 * d * f) + v * d)
    out = []
    for B in (1, 8):
        prompt = torch.randint(0, v, (B, ctx), device=dev)
        model.generate_greedy(prompt[:, :16], 8)  # warm up kernels and buffers
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        model.generate_greedy(prompt, 1)
        torch.cuda.synchronize()
        t_prefill = time.perf_counter() - t0
        t0 = time.perf_counter()
        model.generate_greedy(prompt, steps + 1)
        torch.cuda.synchronize()
        t = (time.perf_counter() - t0 - t_prefill) / steps  # decode steps only (graph capture included)
        by = weight_b + 2.0 * 2 * d * nl * B * (ctx + steps / 2)
        out.append({"batch": B, "context": ctx, "ms_per_step": round(t * 1e3, 4), "tokens_per_s": round(B / t, 1),
                    "prefill_ms": round(t_prefill * 1e3, 1), "step_bytes": int(by), "GBs": round(by / t / 1e9, 1),
                    "frac_of_hbm_peak": round(by / t / 1e9 / HBM_PEAK_GBS, 4)})
    return out


# Shader-clock samples that thread 0 of every workgroup of the batch-1 persistent kernel takes per layer,
# in order (csrc/mega.hip: the stamps in the layer loop, and two inside every gemm_phase).  The kernel has
# no grid barrier inside the layers: a phase's units sit on their own stretch of workgroups and every
# hand-off is polled for, so a step's critical path runs from role to role.
_GEMM = ["activations in LDS -> MFMAs issued", "cross-wave sum"]
PHASE_STAMPS = (
    ["P1 staged"] + ["P1 " + x for x in _GEMM] + ["P1 epilogue", "P2 partials stored", "P2 requests issued", "P3 merged"]
    + ["P3 " + x for x in _GEMM] + ["P3 epilogue", "P4 staged"] + ["P4 " + x for x in _GEMM]
    + ["P4 epilogue", "P4 requests issued", "P5 staged"] + ["P5 " + x for x in _GEMM] + ["P5 epilogue", "P5 requests issued"]
)
PHASE_TAIL = 13  # samples after the layers: three around the final norm, vocabulary projection (2), its end, selection (6), the end


def _polled_roles(cfg, nwg, batch=1):
    """Which workgroups take which phase of the polled builds (mirrors the assignment in csrc/mega_kernel.h)."""
    d, F = cfg.hidden_size, cfg.intermediate_size
    H = cfg.num_attention_heads
    Hkv = cfg.num_key_value_heads or H
    D = d // H
    n_qkv, n_wo, n_dn = (H + 2 * Hkv) * D // 16, d // 16, d // 16
    n_gu = (2 * ((F + 7) // 8 * 8) // 16 + 1) // 2
    chunks = batch * Hkv * max(1, min(16, nwg // (batch * Hkv)))
    dn0 = n_wo if n_wo + n_dn <= nwg else nwg - n_dn
    free = max(dn0 + n_dn, n_gu)
    at0 = free if batch == 1 and nwg - n_qkv - free >= chunks else 0
    return {"qkv": range(nwg - n_qkv, nwg), "attention": range(at0, at0 + min(chunks, nwg)), "merge": range(max(0, nwg - batch * H), nwg),
            "wo": range(0, n_wo), "gate/up": range(0, n_gu), "down": range(dn0, dn0 + n_dn)}


def phase_timeline(dev, prompt_len, steps=32, batch=1, int8=False):
    """The critical path of a layer of the batch-1 persistent kernel: for every hand-off, when the last
    workgroup of the producing role had issued its stores and when the last workgroup of the consuming
    role had the data staged, from the kernel's own clock samples (a 100 MHz counter common to all
    workgroups), averaged over `steps` real decode steps and over the layers after the first."""
    from ohara_amd.llama import Llama

    cfg, st = d12_state(dev)
    model = Llama(cfg, st, device=dev)
    sess = model.session(batch, steps + 24, persistent=True, kv_cache=model.build_kv_cache(batch, int8=True) if int8 else None)
    sess.prefill(torch.randint(0, cfg.vocab_size, (batch, prompt_len)).to(dev))
    for _ in range(8):
        sess.step()
    nl = cfg.num_hidden_layers
    per = len(PHASE_STAMPS)
    roles = _polled_roles(cfg, sess._nwg, batch)
    acc, total_ms = None, 0.0
    for _ in range(steps):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        sess.step(prof_kernel=-2)
        e1.record()
        torch.cuda.synchronize()
        total_ms += e0.elapsed_time(e1)
        c = sess.phase_clocks(None).double()
        c = c - c[:, 0].min()
        acc = c if acc is None else acc + c
    acc = acc / steps / 100.0  # us
    kernel_us = total_ms / steps * 1e3
    idx = {name: j + 1 for j, name in enumerate(PHASE_STAMPS)}  # sample 0 precedes the first layer

    def last(role, name, layer):
        return float(acc[list(roles[role]), layer * per + idx[name]].max())

    chain = [("qkv", "P1 staged", "stream polled for, norm1 in LDS"), ("qkv", "P1 epilogue", "q/k/v product, rotary, q and new k/v rows stored"),
             ("attention", "P2 partials stored", "q polled for, chunk, partials stored"),
             ("merge", "P2 requests issued", "a head's partials polled for and merged (and the next q/k/v weights requested)"),
             ("wo", "P3 merged", "merged rows polled for"), ("wo", "P3 epilogue", "output projection + residual stored"),
             ("gate/up", "P4 staged", "stream polled for, norm2 in LDS"), ("gate/up", "P4 epilogue", "gate/up product, SwiGLU stored"),
             ("down", "P5 staged", "activations polled for, in LDS"), ("down", "P5 epilogue", "down projection + residual stored")]
    seg = torch.zeros(len(chain) + 1, dtype=torch.float64)
    layers = range(1, nl - 1)
    for l in layers:
        t = [last(r, n, l) for r, n, _ in chain] + [last("qkv", "P1 staged", l + 1)]
        prev = last("down", "P5 epilogue", l - 1)
        seg += torch.tensor([t[0] - prev] + [t[i] - t[i - 1] for i in range(1, len(chain))] + [t[-1] - t[0]])
    seg /= len(layers)
    out = {"kernel_us_hip_events (stamps on)": round(kernel_us, 2), "layers": nl, "workgroups": sess._nwg,
           "roles (workgroups)": {k: [v.start, v.stop - 1] for k, v in roles.items()},
           "per_layer_us": round(float(seg[-1]), 3),
           "before_first_layer_us": round(float(acc[list(roles["qkv"]), idx["P1 staged"]].max()), 2),
           "after_last_layer_us (final norm + vocabulary projection + selection)":
               round(float(acc[:, nl * per + PHASE_TAIL].max()) - last("down", "P5 epilogue", nl - 1), 2),
           "critical_path_us (last workgroup of the role, from the previous entry)":
               {f"{r}: {what}": round(float(seg[i]), 3) for i, (r, _, what) in enumerate(chain)}}
    return out


def bitnet_phase_timeline(dev, batch=1, steps=16):
    """Per-phase timeline of the single-launch BitNet decode step (C4 size, context 2047 -> 2048):
    workgroup 0's shader-clock samples at every grid barrier (six per barrier: phase work issued, own
    stores complete, workgroup barrier passed, arrival issued, prefetch issued, barrier passed) or, for
    a single sequence, behind every poll and every phase, averaged over `steps` launches and over the layers after the first."""
    from ohara_amd.bitnet import BitLlama

    cfg, st = bitnet_c4_state(dev)
    model = BitLlama(cfg, st, device=dev)
    del st
    L, nl = cfg.max_sequence_length, cfg.num_hidden_layers
    cache = model.build_kv_cache(batch)
    sess = model.session(batch, 8, kv_cache=cache, persistent=True)
    sess.prefill(torch.randint(0, cfg.vocab_size, (batch, 1), device=dev))
    _fill_cache(cache, L - 1, batch)
    start = torch.tensor([L - 1, 1, 0, 0], dtype=torch.int32, device=dev)
    acc, total_ms = None, 0.0
    for it in range(steps + 4):
        sess.step_state.copy_(start)
        sess._dst.prof_kernel = -2
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        sess._launch_step()
        e1.record()
        torch.cuda.synchronize()
        if it >= 4:
            c = sess.phase_clocks().double()
            acc = c if acc is None else acc + c
            total_ms += e0.elapsed_time(e1)
    sess.check_error()
    c = acc / steps
    kernel_us = total_ms / steps * 1e3
    if batch == 1:  # ten samples a layer (100 MHz clock) of workgroup 0 and, 512 words on, of the first one of the down projection
        first, down = c[: nl * 10].view(nl, 10), c[512 : 512 + nl * 10].view(nl, 10)
        us = lambda t, a, b: round(float((t[1:, b] - t[1:, a]).mean()) / 100, 2)  # noqa: E731
        return {"batch": 1, "kernel_us_hip_events": round(kernel_us, 1), "layers": nl,
                "per_layer_us": round(float((first[1:, 9] - first[:-1, 9]).mean()) / 100, 2),
                "after_last_layer_us (final norm + vocabulary projection + selection)": round(float(c[nl * 10 + 7] - first[-1, 9]) / 100, 1),
                "us": {"stream polled for (q/k/v)": round(float((down[1:, 0] - down[:-1, 9]).mean()) / 100, 2),
                       "q/k/v + rotary + append": us(down, 0, 1), "attention: q polled for, partials": us(down, 1, 2),
                       "merge of a head": us(down, 2, 3), "merged row polled for": us(first, 3, 4), "output projection": us(first, 4, 5),
                       "stream polled for (gate/up)": us(first, 5, 6), "gate/up + SwiGLU": us(first, 6, 7),
                       "activations polled for": us(down, 7, 8), "down projection": us(down, 8, 9)}}
    per = c[: nl * 30].view(nl, 30)
    n_tail = 8  # after the last barrier of the layers: vocabulary projection (2), selection arrive (4) / wait (2)
    ticks_per_us = float(c[nl * 30 + n_tail - 1] - c[0]) / kernel_us  # within a few us of the whole launch
    names = ["P1 q/k/v + rotary + append", "P2 attention partials", "P3 merge + attn.proj + residual",
             "P4 gate/up + SwiGLU", "P5 down (K split in 2)"]
    out = {"batch": batch, "kernel_us_hip_events": round(kernel_us, 1), "layers": nl,
           "clock_ticks_per_us": round(ticks_per_us, 1),
           "per_layer_us": round(float((per[1:, 29] - per[:-1, 29]).mean()) / ticks_per_us, 2),
           "after_last_layer_us (final norm + vocabulary projection + selection)":
               round(float(c[nl * 30 + n_tail - 1] - per[-1, 29]) / ticks_per_us, 1), "phases": {}}
    for i, nm in enumerate(names):
        b = per[1:, i * 6: i * 6 + 6]
        began = per[:-1, 29] if i == 0 else per[1:, i * 6 - 1]
        out["phases"][nm] = {
            "work_us": round(float((b[:, 0] - began).mean()) / ticks_per_us, 2),
            "own_stores_complete_us": round(float((b[:, 1] - b[:, 0]).mean()) / ticks_per_us, 2),
            "workgroup_barrier_us": round(float((b[:, 2] - b[:, 1]).mean()) / ticks_per_us, 2),
            "arrival_us": round(float((b[:, 3] - b[:, 2]).mean()) / ticks_per_us, 2),
            "prefetch_issue_us": round(float((b[:, 4] - b[:, 3]).mean()) / ticks_per_us, 2),
            "wait_for_release_us": round(float((b[:, 5] - b[:, 4]).mean()) / ticks_per_us, 2)}
    return out


HYBRID_SIZES = {"d1024": (1024, 8, 8, 4, 128, 2816), "d2048": (2048, 8, 16, 4, 128, 5632)}  # width, layers, heads, KV heads, head size, ff


def hybrid_llama(name, dev):
    """A Llama of a size's width, depth, heads and feed-forward with random weights."""
    from ohara_amd.llama import Config, Llama

    d, layers, H, G, dh, ff = HYBRID_SIZES[name]
    cfg = Config(vocab_size=32000, hidden_size=d, intermediate_size=ff, num_attention_heads=H, num_key_value_heads=G,
                 num_hidden_layers=layers, dropout=0.0, max_sequence_length=4608)
    g = torch.Generator(device=dev).manual_seed(0)
    n = lambda *shape: (torch.randn(*shape, generator=g, device=dev) * 0.02).to(torch.bfloat16)  # noqa: E731
    one = torch.ones(d, dtype=torch.bfloat16, device=dev)
    st = {"token_emb.weight": n(32000, d), "vocab_proj.weight": n(32000, d), "norm.weight": one}
    for i in range(layers):
        p = f"layers.{i}."
        st.update({p + "attn.query.weight": n(d, d), p + "attn.key.weight": n(G * dh, d), p + "attn.value.weight": n(G * dh, d),
                   p + "attn.proj.weight": n(d, d), p + "ff.up.weight": n(ff, d), p + "ff.gate.weight": n(ff, d),
                   p + "ff.down.weight": n(d, ff), p + "norm1.weight": one, p + "norm2.weight": one})
    return Llama(cfg, st, device=dev)


def povazen_size(name):
    """The config dict of the hybrid model."""
    d, n, H, G, dh, ff = HYBRID_SIZES[name]
    mlp = {"kind": "dense", "ff": ff}
    delta = {"type": "channel_delta", "mixer": {"heads": H, "kv_heads": H, "dim": dh, "vdim": dh, "conv": 4}, "mlp": mlp}
    att = {"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": dh, "vdim": dh, "scale": dh ** -0.5}, "mlp": mlp}
    return {"width": d, "vocab": 32000, "canon": {"taps": 4}, "norm": {"eps": 1e-6, "groups": 1}, "logit_softcap": 30.0,
            "layers": ([delta] * 3 + [att]) * (n // 4)}


def povazen_state(cfg, dev, rank=128, seed=5):
    """Random weights of a hybrid config: matrices N(0, 1/columns), unit norms, decays of some tens of tokens."""
    g = torch.Generator(device=dev).manual_seed(seed)
    n = lambda *shape, s=1.0: (torch.randn(*shape, generator=g, device=dev) * s).to(torch.bfloat16)  # noqa: E731
    lin = lambda o, i: n(o, i, s=i ** -0.5)  # noqa: E731
    one = lambda k: torch.ones(k, device=dev, dtype=torch.bfloat16)  # noqa: E731
    d = cfg["width"]
    st = {"embed": n(cfg["vocab"], d), "head": lin(cfg["vocab"], d), "final.norm": one(d)}
    for i, layer in enumerate(cfg["layers"]):
        p, m, ff = f"l{i}.", layer["mixer"], layer["mlp"]["ff"]
        H, K, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        st.update({p + "norm1": one(d), p + "norm2": one(d), p + "canon1": n(d, cfg["canon"]["taps"], s=0.2),
                   p + "mlp.gate": lin(ff, d), p + "mlp.up": lin(ff, d), p + "mlp.down": lin(d, ff)})
        p += "mix."
        st.update({p + "k": lin(K * D, d), p + "o": lin(d, H * V)})
        if layer["type"] == "attention":
            st.update({p + "q": lin(H * D, d), p + "v": lin(K * V, d), p + "q.b": n(H * D, s=0.1), p + "k.b": n(K * D, s=0.1),
                       p + "v.b": n(K * V, s=0.1), p + "q.norm": one(H * D), p + "k.norm": one(K * D), p + "g": lin(H, d)})
        else:
            st.update({p + "q": lin(K * D, d), p + "v": lin(H * V, d), p + "b": lin(H, d), p + "norm": one(V),
                       p + "A_log": torch.zeros(H, device=dev, dtype=torch.bfloat16), p + "dt_bias": n(H * D) - 3.0,
                       p + "a1": lin(rank, d), p + "a2": lin(H * D, rank), p + "g1": lin(rank, d), p + "g2": lin(H * V, rank)})
            for c, k in (("q", K * D), ("k", K * D), ("v", H * V)):
                st[p + c + ".conv"] = n(k, m["conv"], s=0.5)
    return st


def _time_model_prefill(model, B, S, dev, reps=3):
    ids = torch.randint(0, model.config.vocab_size, (B, S), device=dev)
    cache = model.build_kv_cache(B)
    best = None
    for _ in range(reps + 1):
        for c in cache:
            c.length, c.batch_size, c.lengths = 0, None, None
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        model(ids, cache, 0, last_only=True)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        best = dt if best is None else min(best, dt)
    return {"ms": round(best * 1e3, 3), "tokens_per_s": round(B * S / best, 1)}


def _time_model_decode(model, B, context, steps=64):
    sess = model.session(B, steps + 32)
    sess.prefill(torch.randint(0, model.config.vocab_size, (B, context)))
    sess.capture()
    sess.run(8)
    torch.cuda.synchronize()
    best = None
    for _ in range(2):
        t0 = time.perf_counter()
        sess.run(steps // 4)
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t0) / (steps // 4)
        best = dt if best is None else min(best, dt)
    sess.check_error()
    return {"ms_per_step": round(best * 1e3, 4), "tokens_per_s": round(B / best, 1)}


FP32_MFMA_PEAK_TFLOPS = 157.3


def _hbm(t, by):
    return {"us": round(t * 1e6, 1), "GBs": round(by / t / 1e9, 1), "frac_of_hbm_peak": round(by / t / 1e9 / HBM_PEAK_GBS, 4)}


def _flops(t, fl, peak):
    return {"us": round(t * 1e6, 1), "TFLOPs": round(fl / t / 1e12, 1), "frac_of_peak": round(fl / t / 1e12 / peak, 4)}


def bench_povazen_kernels(cfg, dev):
    """The hybrid model's own kernels beside the like kernels of Llama at one layer's sizes."""
    from ohara_amd import ops
    from ohara_amd.hybrid import distance_slopes
    from ohara_amd.povazen import Povazen, PovazenConfig

    bf = torch.bfloat16
    model = Povazen(PovazenConfig.from_dict({**cfg, "layers": cfg["layers"][2:4]}, 4096),
                    {k.replace("l2.", "l0.").replace("l3.", "l1."): v for k, v in povazen_state(cfg, dev).items()
                     if not k.startswith(("l0.", "l1."))}, device=dev)
    delta, att = (b["mixer"] for b in model.layers)
    H, G, D, V, d = att.heads, att.kv_heads, att.dim, att.vdim, cfg["width"]
    slopes = distance_slopes(H).to(dev)
    rnd = lambda *shape, dt=bf: torch.randn(*shape, device=dev).to(dt)  # noqa: E731
    rows = []

    def timed(fn, n=8):  # n calls per graph: what a single-launch graph costs to start would swamp the small kernels
        return graph_time(lambda: [fn() for _ in range(n)], iters=20) / n

    for B, L in ((1, 4096), (8, 4096), (32, 2048)):
        q, k, v = rnd(B, H * D), rnd(B, L, G, D), rnd(B, L, G, V)
        ns = att.n_split(B, L)
        ws = ops.attn_bias_workspace(B, H, V, ns, dev)
        gate = rnd(B, H)
        seq = ops.Seq(B, 1, L - 1)
        by = 2.0 * G * (D + V) * B * L
        row = {"kernel": "decode attention", "batch": B, "context": L,
               "attn_bias_kernel": _hbm(timed(lambda: ops.attn_bias(q, k, v, H, G, D, V, 0.1, slopes, gate, seq, ns, ws)), by)}
        n2 = max(1, min(1024 // (B * G), L // 128, 64))
        ws2 = ops.attn_workspace(B, H, G, D, n2, dev)
        row["llama attn_decode_kernel"] = _hbm(timed(lambda: ops.attn_decode(q, k, v, H, G, D, L, n2, ws2)), by)
        rows.append(row)
    for B, S in ((1, 4096), (8, 1024)):
        q, k, v = rnd(B * S, H * D), rnd(B, S, G, D), rnd(B, S, G, V)
        gate = rnd(B * S, H)
        seq = ops.Seq(B, S, 0)
        fl = 2.0 * B * H * (D + V) * S * (S + 1) / 2
        rows.append({"kernel": "prompt attention", "batch": B, "tokens": S,
                     "attn_bias_prefill_kernel": _flops(timed(lambda: ops.attn_bias(q, k, v, H, G, D, V, 0.1, slopes, gate, seq)),
                                                        fl, MFMA_BF16_PEAK_TFLOPS),
                     "llama attn_prefill": _flops(timed(lambda: ops.attn_prefill(q, k, v, H, G, D, 0, S)), fl,
                                                         MFMA_BF16_PEAK_TFLOPS)})
    x = rnd(1, 2048)
    wn = torch.ones(2048, device=dev, dtype=bf)
    base = _hbm(timed(lambda: ops.rmsnorm(x, wn)), 2.0 * 2 * 2048)
    for B in (1, 8, 32):
        st = delta.state(B, 4096)
        p = rnd(B, delta.proj.n)
        seq = ops.Seq(B, 1, 100)
        h = delta.heads
        by = 2.0 * 4 * B * h * delta.dim * delta.vdim + 2.0 * (delta.a2.numel() + delta.g2.numel())
        row = {"kernel": "delta rule, one token", "batch": B,
               "delta_step_kernel": _hbm(timed(lambda: ops.delta_step(delta._c, p, st["delta"], st["ring"], seq)), by)}
        xf, y = rnd(B, d, dt=torch.float32), rnd(B, d)
        blk = model.layers[0]
        ring = blk["conv"].state(B)
        row["residual_norm_kernel (norm, residual, convolution)"] = _hbm(timed(lambda: ops.residual_norm(
            xf, seq, bf, y=y, norm_w=blk["norm1"].w, groups=1, eps=1e-6, mode="conv", conv_w=blk["conv"].w, ring=ring)),
            B * d * (8.0 + 2 + 2 + 4 * 4 + 4))
        row["llama rmsnorm_kernel, one row"] = base
        rows.append(row)
    for B, S in ((1, 4096), (8, 1024)):
        st = delta.state(B, 4096)
        p = rnd(B * S, delta.proj.n)
        za, zg = rnd(B * S, delta.heads * delta.dim) - 3.0, rnd(B * S, delta.heads * delta.vdim)
        ws = delta._workspace(B, S)
        seq = ops.Seq(B, S, 0)
        t = timed(lambda: ops.delta_prefill(delta._c, p, za, zg, st["delta"], st["ring"], ws, seq))
        # the recurrence's own work: decay, two products with the state and the write, per token and head
        fl = 7.0 * B * S * delta.heads * delta.dim * delta.vdim
        xf, y = rnd(B * S, d, dt=torch.float32), rnd(B * S, d)
        blk = model.layers[0]
        ring = blk["conv"].state(B)
        tn = timed(lambda: ops.residual_norm(xf, seq, bf, y=y, norm_w=blk["norm1"].w, groups=1, eps=1e-6, mode="none"))
        tc = timed(lambda: ops.input_conv(xf, blk["conv"].w, ring, seq, bf))
        tr = timed(lambda: ops.rmsnorm(y, blk["norm1"].w.to(bf)))
        big = rnd(B * S, att.proj.n)
        kc, vc = rnd(B, S, G, D), rnd(B, S, G, V)
        tq = timed(lambda: ops.qkv_norm_append(big, H, G, D, V, att.q_norm, att.k_norm, 1e-6, kc, vc, seq))
        rows.append({"kernel": "delta rule, prompt", "batch": B, "tokens": S, "delta_prefill (3 kernels)": _flops(t, fl, FP32_MFMA_PEAK_TFLOPS),
                     "residual_norm_kernel": _hbm(tn, B * S * d * 10.0), "input_conv_kernel + ring": _hbm(tc, B * S * d * 6.0),
                     "qkv_norm_append_kernel": _hbm(tq, 4.0 * B * S * (H * D + G * (D + V))),
                     "llama rmsnorm_kernel": _hbm(tr, B * S * d * 4.0)})
    return rows


def bench_models(name, models, dev):
    """Prefill and decode figures of (label, constructor) pairs, one model in memory at a time."""
    out = {}
    for label, make in models:
        model = make()
        out[label] = {"parameters": sum(t.numel() for t in model.parameters()),
                      "prefill": {f"{B}x{S}": _time_model_prefill(model, B, S, dev) for B, S in ((1, 512), (1, 4096), (8, 1024))},
                      "decode": {f"batch {B}, context {L}": _time_model_decode(model, B, L)
                                 for B, L in ((1, 1024), (1, 4096), (8, 4096), (32, 2048))}}
        del model
        torch.cuda.empty_cache()
    return out


def bench_povazen(dev, sizes=("d1024", "d2048"), kernels=True):
    """Prefill and decode of the hybrid model (three delta-rule layers to one attention layer, SwiGLU everywhere, random
    weights) beside Llama at the same width, depth, heads and feed-forward."""
    from ohara_amd.povazen import Povazen, PovazenConfig

    out = {}
    for name in sizes:
        cfg = povazen_size(name)
        out[name] = {"layers": len(cfg["layers"]), "width": cfg["width"], **bench_models(name, (
            ("povazen", lambda: Povazen(PovazenConfig.from_dict(cfg, 4608), povazen_state(cfg, dev), device=dev)),
            ("llama", lambda: hybrid_llama(name, dev))), dev)}
        if kernels:
            out[name]["kernels"] = bench_povazen_kernels(cfg, dev)
    return out


def vavelorn_size(name):
    """The config dict: two delta-rule layers to one of latent and one of chunked rotary attention."""
    d, n, H, G, dh, ff = HYBRID_SIZES[name]
    layer = lambda kind, **m: {"type": kind, "mixer": {"heads": H, "dim": dh, "vdim": dh, **m}, "mlp": {"kind": "dense", "ff": ff}}  # noqa: E731
    delta = layer("delta", kv_heads=H, conv=4)
    latent = layer("latent_attention", kv_rank=512, q_rank=d // 2, scale=dh ** -0.5)
    att = layer("attention", kv_heads=G, scale=dh ** -0.5, rot={"base": 1e4, "dims": dh // 2}, softcap=30.0, mask={"size": 4096})
    return {"width": d, "vocab": 32000, "token_side": {"dim": 64}, "norm": {"eps": 1e-5}, "layers": [delta, latent, delta, att] * (n // 4)}


def vavelorn_state(cfg, dev, seed=5):
    """Random weights: matrices N(0, 1/columns), unit norms, decays of some tens of tokens."""
    g = torch.Generator(device=dev).manual_seed(seed)
    n = lambda *shape, s=1.0: (torch.randn(*shape, generator=g, device=dev) * s).to(torch.bfloat16)  # noqa: E731
    lin = lambda o, i: n(o, i, s=i ** -0.5)  # noqa: E731
    one = lambda k: torch.ones(k, device=dev, dtype=torch.bfloat16)  # noqa: E731
    d, side = cfg["width"], cfg["token_side"]["dim"]
    st = {"embed": n(cfg["vocab"], d), "side.embed": n(cfg["vocab"], side * len(cfg["layers"])), "head": lin(cfg["vocab"], d),
          "final.norm": one(d)}
    for i, layer in enumerate(cfg["layers"]):
        p, m, ff = f"l{i}.", layer["mixer"], layer["mlp"]["ff"]
        H, K, D, V = m["heads"], m.get("kv_heads"), m["dim"], m["vdim"]
        st.update({p + f"norm{k}": one(d) for k in ("1", "1b", "2", "2b")})
        st.update({p + "mlp.gate": lin(ff, d), p + "mlp.up": lin(ff, d), p + "mlp.down": lin(d, ff), p + "side.gate": lin(side, d),
                   p + "side.proj": lin(d, side), p + "side.norm": one(d)})
        p += "mix."
        st[p + "o"] = lin(d, H * V)
        if layer["type"] == "latent_attention":
            r, rq = m["kv_rank"], m["q_rank"]
            st.update({p + "dq": lin(rq, d), p + "dq.norm": one(rq), p + "uq": lin(H * D, rq), p + "dkv": lin(r, d), p + "dkv.norm": one(r),
                       p + "uk": lin(H * D, r), p + "uv": lin(H * V, r), p + "g": lin(H * V, d)})
            continue
        vrows = K * V if layer["type"] == "attention" else H * V
        st.update({p + "q": lin(H * D if layer["type"] == "attention" else K * D, d), p + "k": lin(K * D, d), p + "v": lin(vrows, d)})
        if layer["type"] == "delta":
            st.update({p + "b": lin(H, d), p + "a": lin(H, d), p + "g": lin(H * V, d), p + "norm": one(V), p + "dt_bias": n(H) - 3.0,
                       p + "A_log": torch.zeros(H, device=dev, dtype=torch.bfloat16)})
            for c, k in (("q", K * D), ("k", K * D), ("v", H * V)):
                st[p + c + ".conv"] = n(k, m["conv"], s=0.5)
    return st


def _sole_layers(build, config_of, state, cfg, kinds, dev):
    """The mixers of the first layer of each kind, from a model of just those layers."""
    at = [next(i for i, layer in enumerate(cfg["layers"]) if layer["type"] == kind) for kind in kinds]
    names = {f"l{i}.": f"l{k}." for k, i in enumerate(at)}
    if "side.embed" in state:
        side = cfg["token_side"]["dim"]
        state = {**state, "side.embed": state["side.embed"][:, :side * len(at)]}
    keep = {names.get(k.split(".")[0] + ".", "") + (k.split(".", 1)[1] if k.split(".")[0] + "." in names else k): v for k, v in state.items()
            if k.split(".")[0] + "." in names or not k.startswith("l")}
    return build(config_of({**cfg, "layers": [cfg["layers"][i] for i in at]}, 4096), keep, device=dev)


def bench_vavelorn_kernels(name, dev):
    """The design's own kernels at one layer's sizes, each beside the like kernel of Llama or Povazen."""
    from ohara_amd import ops
    from ohara_amd.hybrid import distance_slopes
    from ohara_amd.povazen import Povazen, PovazenConfig
    from ohara_amd.vavelorn import Vavelorn, VavelornConfig

    bf, cfg, pcfg = torch.bfloat16, vavelorn_size(name), povazen_size(name)
    model = _sole_layers(Vavelorn, VavelornConfig.from_dict, vavelorn_state(cfg, dev), cfg, ("delta", "latent_attention", "attention"), dev)
    pov = _sole_layers(Povazen, PovazenConfig.from_dict, povazen_state(pcfg, dev), pcfg, ("channel_delta", "attention"), dev)
    delta, lat, att = (b["mixer"] for b in model.layers)
    pdelta, patt = (b["mixer"] for b in pov.layers)
    H, G, D, V, d, R = att.heads, att.kv_heads, att.dim, att.vdim, cfg["width"], lat.rank
    slopes = distance_slopes(H).to(dev)
    rnd = lambda *shape, dt=bf: torch.randn(*shape, device=dev).to(dt)  # noqa: E731
    rows = []

    def timed(fn, n=8):  # n calls per graph: what a single-launch graph costs to start would swamp the small kernels
        return graph_time(lambda: [fn() for _ in range(n)], iters=20) / n

    for B, L in ((1, 4096), (8, 4096), (32, 2048)):
        seq = ops.Seq(B, 1, L - 1)
        q, k, v = rnd(B, H * D), rnd(B, L, G, D), rnd(B, L, G, V)
        ns, ws = att._split(B, L)
        t_att = timed(lambda: ops.attn_scored(q, k, v, H, G, D, V, L, 0.1, seq, cap=30.0, chunk=4096, n_split=ns, workspace=ws))
        n2 = max(1, min(1024 // (B * G), L // 128, 64))
        ws2 = ops.attn_workspace(B, H, G, D, n2, dev)
        t_llama = timed(lambda: ops.attn_decode(q, k, v, H, G, D, L, n2, ws2))
        by = 2.0 * G * (D + V) * B * L
        c, ql = rnd(B, L, R), rnd(B, H * R)
        nl, wl = lat._split(B, L)
        t_lat = timed(lambda: ops.attn_latent(ql, c, H, R, 0.1, seq, nl, wl))
        rows.append({"kernel": "decode attention", "batch": B, "context": L, "attn_bias_kernel (cap, chunk)": _hbm(t_att, by),
                     "llama attn_decode_kernel": _hbm(t_llama, by), "attn_latent_kernel + merge": _hbm(t_lat, 2.0 * R * B * L)})
    for B, S in ((1, 4096), (8, 1024)):
        seq = ops.Seq(B, S, 0)
        q, k, v = rnd(B * S, H * D), rnd(B, S, G, D), rnd(B, S, G, V)
        fl = 2.0 * B * H * (D + V) * S * (S + 1) / 2
        gate, ge, kv = rnd(B * S, H), rnd(B * S, H * V), rnd(B * S, H * (D + V))
        rows.append({
            "kernel": "prompt attention", "batch": B, "tokens": S,
            "attn_bias_prefill_kernel (cap, chunk)": _flops(timed(lambda: ops.attn_scored(
                q, k, v, H, G, D, V, S, 0.1, seq, cap=30.0, chunk=4096)), fl, MFMA_BF16_PEAK_TFLOPS),
            "latent: attn_bias_prefill_kernel (expanded, gated)": _flops(timed(lambda: ops.attn_scored(
                q, kv, kv[:, H * D:], H, H, D, V, S, 0.1, seq, gate=ge, gate_elements=True, ld_k=H * (D + V), ld_v=H * (D + V))), fl,
                MFMA_BF16_PEAK_TFLOPS),
            "povazen attn_bias_prefill_kernel": _flops(timed(lambda: ops.attn_bias(q, k, v, H, G, D, V, 0.1, slopes, gate, seq)), fl,
                                                       MFMA_BF16_PEAK_TFLOPS),
            "llama attn_prefill": _flops(timed(lambda: ops.attn_prefill(q, k, v, H, G, D, 0, S)), fl, MFMA_BF16_PEAK_TFLOPS)})
    side, norm, after = model.layers[0]["side"], model.layers[0]["norm2b"], model.layers[1]["norm1"]
    plain = ops.pack_linear(rnd(side.gate.n, d))
    for B in (1, 8, 32):
        seq, ids = ops.Seq(B, 1, 100), torch.randint(0, 32000, (B,), device=dev)
        row = {"kernel": "one token", "batch": B}
        for label, mix, more in (("delta_step_kernel", delta, 2.0 * B * H * V),
                                 ("povazen delta_step_kernel", pdelta, 2.0 * (pdelta.a2.numel() + pdelta.g2.numel()))):
            st, p = mix.state(B, 4096), rnd(B, mix.proj.n)
            row[label] = _hbm(timed(lambda: ops.delta_step(mix._c, p, st["delta"], st["ring"], seq)), 8.0 * B * H * D * V + more)
        x, xl, gate = rnd(B, H * D), rnd(B, H * R), rnd(B, H * V)
        by = 2.0 * H * R * D
        row["head_linear_kernel (keys)"] = _hbm(timed(lambda: ops.head_linear(x, lat.k_absorb, R)), by)
        row["head_linear_kernel (values, gate)"] = _hbm(timed(lambda: ops.head_linear(xl, lat.v_absorb, V, gate)), by)
        w = ops.pack_linear(rnd(R * 2, H * D // 2))
        xs = rnd(B, H * D // 2)
        row["llama gemm_skinny, as many weights"] = _hbm(timed(lambda: ops.gemm_skinny(xs, w)), by)
        hx = rnd(B, d)
        row["gemm_gelu_lookup"] = _hbm(timed(lambda: ops.gemm_gelu_lookup(hx, side.gate.w, side.table, 0, ids)), 2.0 * side.gate.n * d)
        row["llama gemm_skinny, same weights"] = _hbm(timed(lambda: ops.gemm_skinny(hx, plain)), 2.0 * side.gate.n * d)
        xf, y = rnd(B, d, dt=torch.float32), rnd(B, d)
        row["residual_norm_kernel (two layer norms)"] = _hbm(timed(lambda: ops.residual_norm(
            xf, seq, bf, **{**norm.of(y), **norm.out()})), B * d * 12.0)
        row["povazen residual_norm_kernel (two norms)"] = _hbm(timed(lambda: ops.residual_norm(
            xf, seq, bf, y=y, norm_w=norm.w, groups=1, eps=1e-5, mode="norm", norm2_w=norm.w)), B * d * 12.0)
        row["token_side_kernel (update, side embedding, norm)"] = _hbm(timed(lambda: ops.token_side(
            xf, y, norm.w, side.gate.w, side.proj.w, side.table, side.column, ids, side.norm.w, norm.eps, after.w, center_y=True,
            center_out=True)),
                                                                      B * d * 12.0 + 4.0 * side.gate.n * d)
        row["the same unfused (4 launches)"] = _hbm(timed(lambda: (
            ops.residual_norm(xf, seq, bf, **{**side.norm.of(side(ops.residual_norm(xf, seq, bf, **{**norm.of(y), "mode": "copy"}), ids)),
                                              **after.out()}))), B * d * 12.0 + 4.0 * side.gate.n * d)
        rows.append(row)
    for B, S in ((1, 4096), (8, 1024)):
        seq, n, ids = ops.Seq(B, S, 0), B * S, torch.randint(0, 32000, (B * S,), device=dev)
        row = {"kernel": "prompt, other kernels", "batch": B, "tokens": S}
        for label, mix in (("delta_prefill (3 kernels)", delta), ("povazen delta_prefill (3 kernels)", pdelta)):
            st, p = mix.state(B, 4096), rnd(n, mix.proj.n)
            za, zg = (None, None) if mix is delta else (rnd(n, H * D) - 3.0, rnd(n, H * V))
            ws = mix._workspace(B, S)
            row[label] = _flops(timed(lambda: ops.delta_prefill(mix._c, p, za, zg, st["delta"], st["ring"], ws, seq)),
                                7.0 * n * H * D * V, FP32_MFMA_PEAK_TFLOPS)
        kc, vc, big = rnd(B, S, G, D), rnd(B, S, G, V), rnd(n, max(att.proj.n, patt.proj.n, lat.proj.n))
        cos, sin = (torch.ones(S, D // 4, device=dev) for _ in range(2))
        by = 4.0 * n * (H * D + G * (D + V))
        row["qkv_rotate_append_kernel"] = _hbm(timed(lambda: ops.qkv_rotate_append(big, H, G, D, V, cos, sin, D // 2, kc, vc, seq)), by)
        row["povazen qkv_norm_append_kernel"] = _hbm(timed(lambda: ops.qkv_norm_append(
            big, H, G, D, V, patt.q_norm, patt.k_norm, 1e-6, kc, vc, seq)), by)
        cl = rnd(B, S, R)
        row["latent_front_kernel"] = _hbm(timed(lambda: ops.latent_front(
            big, lat.q_rank, lat.off_c, R, lat.q_norm, lat.kv_norm, 1e-5, cl, seq, True)), 2.0 * n * (2 * lat.q_rank + 3 * R))
        hx = rnd(n, d)
        fl = 2.0 * n * side.gate.n * d
        row["gemm_gelu_lookup"] = _flops(timed(lambda: ops.gemm_gelu_lookup(hx, side.gate.w, side.table, 0, ids)), fl, MFMA_BF16_PEAK_TFLOPS)
        row["llama gemm, same weights"] = _flops(timed(lambda: ops.gemm_skinny(hx, plain)), fl, MFMA_BF16_PEAK_TFLOPS)
        xf, y = rnd(n, d, dt=torch.float32), rnd(n, d)
        row["residual_norm_kernel (two layer norms)"] = _hbm(timed(lambda: ops.residual_norm(
            xf, seq, bf, **{**norm.of(y), **norm.out()})), n * d * 12.0)
        row["povazen residual_norm_kernel (two norms)"] = _hbm(timed(lambda: ops.residual_norm(
            xf, seq, bf, y=y, norm_w=norm.w, groups=1, eps=1e-5, mode="norm", norm2_w=norm.w)), n * d * 12.0)
        row["token_side_kernel (update, side embedding, norm)"] = _hbm(timed(lambda: ops.token_side(
            xf, y, norm.w, side.gate.w, side.proj.w, side.table, side.column, ids, side.norm.w, norm.eps, after.w, center_y=True,
            center_out=True)),
                                                                      n * d * 12.0 + 4.0 * side.gate.n * d)
        row["the same unfused (4 launches)"] = _hbm(timed(lambda: (
            ops.residual_norm(xf, seq, bf, **{**side.norm.of(side(ops.residual_norm(xf, seq, bf, **{**norm.of(y), "mode": "copy"}), ids)),
                                              **after.out()}))), n * d * 12.0 + 4.0 * side.gate.n * d)
        rows.append(row)
    return rows


def bench_vavelorn(dev, sizes=("d1024", "d2048")):
    """Prefill and decode of Vavelorn with random weights beside Povazen and Llama at the same width, depth, heads and feed-forward."""
    from ohara_amd.povazen import Povazen, PovazenConfig
    from ohara_amd.vavelorn import Vavelorn, VavelornConfig

    out = {}
    for name in sizes:
        cfg, pcfg = vavelorn_size(name), povazen_size(name)
        out[name] = {"layers": len(cfg["layers"]), "width": cfg["width"], **bench_models(name, (
            ("vavelorn", lambda: Vavelorn(VavelornConfig.from_dict(cfg, 4608), vavelorn_state(cfg, dev), device=dev)),
            ("povazen", lambda: Povazen(PovazenConfig.from_dict(pcfg, 4608), povazen_state(pcfg, dev), device=dev)),
            ("llama", lambda: hybrid_llama(name, dev))), dev)}
        out[name]["kernels"] = bench_vavelorn_kernels(name, dev)
    return out


FIBIRAX_EXPERTS = (28, 4, 4, 4, 2)  # experts, identity outputs, used per token, groups, groups kept


def fibirax_size(name):
    """The config dict: attention in a window of 1024 beside retention in every layer, four of 28 experts (and four identity
    outputs) of an eighth of the feed-forward and a shared one of half of it."""
    d, n, H, G, dh, ff = HYBRID_SIZES[name]
    experts, identity, top, groups, keep = FIBIRAX_EXPERTS
    left = {"heads": H, "kv_heads": G, "dim": dh, "vdim": dh, "scale": dh ** -0.5, "softcap": 30.0, "mask": {"size": 1024},
            "rot": {"base": 5e5, "dims": dh, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    right = {"heads": H, "dim": dh, "vdim": dh, "decay": [1 - 2.0 ** (-5 - 7 * h / H) for h in range(H)]}
    mlp = {"kind": "moe", "router": {"experts": experts, "identity": identity, "top": top, "groups": {"count": groups, "keep": keep}},
           "expert": {"ff": ff // 8, "limit": 7.0}, "shared": {"ff": ff // 2, "limit": 7.0}}
    one = {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0}, "mlp": mlp}
    return {"width": d, "vocab": 32000, "embedding": {"scale": d ** 0.5}, "norm": {"eps": 1e-6}, "layers": [one] * n}


def fibirax_state(cfg, dev, seed=5):
    """Random weights: matrices N(0, 1/columns), unit norms, corrections of a tenth of a score."""
    g = torch.Generator(device=dev).manual_seed(seed)
    n = lambda *shape, s=1.0: (torch.randn(*shape, generator=g, device=dev) * s).to(torch.bfloat16)  # noqa: E731
    lin = lambda o, i: n(o, i, s=i ** -0.5)  # noqa: E731
    one = lambda k: torch.ones(k, device=dev, dtype=torch.bfloat16)  # noqa: E731
    d = cfg["width"]
    st = {"embed": n(cfg["vocab"], d), "head": lin(cfg["vocab"], d), "final.norm": one(d)}
    for i, layer in enumerate(cfg["layers"]):
        p, a, r, mlp = f"l{i}.", layer["mixer"]["left"], layer["mixer"]["right"], layer["mlp"]
        st.update({p + k: one(d) for k in ("norm1", "norm2", "ls1", "ls2")})
        q = p + "mix.left."
        st.update({q + "q": lin(a["heads"] * a["dim"], d), q + "k": lin(a["kv_heads"] * a["dim"], d), q + "v": lin(a["kv_heads"] * a["vdim"], d),
                   q + "o": lin(d, a["heads"] * a["vdim"]), q + "q.norm": one(a["dim"]), q + "k.norm": one(a["dim"])})
        q = p + "mix.right."
        nk, nv = r["heads"] * r["dim"], r["heads"] * r["vdim"]
        st.update({q + "q": lin(nk, d), q + "k": lin(nk, d), q + "v": lin(nv, d), q + "g": lin(nv, d), q + "o": lin(d, nv)})
        q, total = p + "mlp.", mlp["router"]["experts"] + mlp["router"]["identity"]
        st.update({q + "router": lin(total, d), q + "correction": n(total, s=0.1 / total)})
        for name, ff in [(f"e{e}", mlp["expert"]["ff"]) for e in range(mlp["router"]["experts"])] + [("shared", mlp["shared"]["ff"])]:
            st.update({f"{q}{name}.gate": lin(ff, d), f"{q}{name}.up": lin(ff, d), f"{q}{name}.down": lin(d, ff)})
    return st


def _like_grouped_moe(name, dev):
    """A Llama's grouped mixture of experts of the same sizes (every output an expert, four of them per token, one shared expert)."""
    from ohara_amd.moe import GroupedMoE

    d, _, _, _, _, ff = HYBRID_SIZES[name]
    E, f, fs = sum(FIBIRAX_EXPERTS[:2]), ff // 8, ff // 2
    g = torch.Generator(device=dev).manual_seed(6)
    n = lambda *shape: (torch.randn(*shape, generator=g, device=dev) * d ** -0.5).to(torch.bfloat16)  # noqa: E731
    return GroupedMoE(n(E, d, f), n(E, d, f), n(E, f, d), n(E, d), torch.zeros(E, device=dev), FIBIRAX_EXPERTS[2],
                      shared=(n(fs, d), n(fs, d), n(d, fs)), device=dev)


def bench_fibirax_kernels(name, dev):
    """The design's own kernels at one layer's sizes, each beside the like kernel of Vavelorn or of Llama's experts."""
    from ohara_amd import ops
    from ohara_amd.fibirax import Fibirax, FibiraxConfig
    from ohara_amd.vavelorn import Vavelorn, VavelornConfig

    bf, cfg, vcfg = torch.bfloat16, fibirax_size(name), vavelorn_size(name)
    cfg = {**cfg, "layers": cfg["layers"][:1]}
    model = Fibirax(FibiraxConfig.from_dict(cfg, 4096), fibirax_state(cfg, dev), device=dev)
    vav = _sole_layers(Vavelorn, VavelornConfig.from_dict, vavelorn_state(vcfg, dev), vcfg, ("delta",), dev)
    like = _like_grouped_moe(name, dev)
    block, delta = model.layers[0], vav.layers[0]["mixer"]
    mixer, experts, norm = block["mixer"], block["mlp"], block["norm2"]
    att, ret = (part for _, part in mixer.parts)
    H, G, D, V, d, W = att.heads, att.kv_heads, att.dim, att.vdim, cfg["width"], att.window
    top, ff, ffs, E = experts.top, experts.ff, experts.shared.ff, experts.experts
    rnd = lambda *shape, dt=bf: torch.randn(*shape, device=dev).to(dt)  # noqa: E731
    rows = []

    def timed(fn, n=8):  # n calls per graph: what a single-launch graph costs to start would swamp the small kernels
        return graph_time(lambda: [fn() for _ in range(n)], iters=20) / n

    for B, L in ((1, 4096), (8, 4096), (32, 2048)):
        seq = ops.Seq(B, 1, L - 1)
        q, k, v = rnd(B, H * D), rnd(B, L, G, D), rnd(B, L, G, V)
        ns, ws = att._split(B, L)
        by = 2.0 * G * (D + V) * B * W
        big, buf, cos, sin = rnd(B, mixer.proj.n), rnd(B, 2 * H * D), *(torch.ones(L, D // 2, device=dev) for _ in range(2))
        small = 4.0 * B * (H * D + G * (D + V))
        rows.append({
            "kernel": "decode attention", "batch": B, "context": L, "window": W,
            "attn_bias_kernel (window, cap, sink)": _hbm(timed(lambda: ops.attn_scored(
                q, k, v, H, G, D, V, L, 0.1, seq, cap=30.0, window=W, sinks=att.sinks, n_split=ns, workspace=ws)), by),
            "vavelorn attn_bias_kernel (chunk, cap)": _hbm(timed(lambda: ops.attn_scored(
                q, k, v, H, G, D, V, L, 0.1, seq, cap=30.0, chunk=W, n_split=ns, workspace=ws)), by),
            "qkv_headnorm_rotate_append_kernel": _hbm(timed(lambda: ops.qkv_headnorm_rotate_append(
                big, H, G, D, V, att.q_norm, att.k_norm, 1e-6, cos, sin, D, k, v, seq)), small),
            "vavelorn qkv_rotate_append_kernel": _hbm(timed(lambda: ops.qkv_rotate_append(big, H, G, D, V, cos, sin, D, k, v, seq)), small)})
        row, st, rst = {"kernel": "recurrence, one token", "batch": B}, delta.state(B, 4096), ret.state(B, 4096)["retention"]
        p, dst = big[:, mixer.n_in:], buf[:, mixer.n_out:mixer.n_out + H * V]
        row["retention_step_kernel"] = _hbm(timed(lambda: ops.retention(ret._c, p, rst, None, seq, dst)), 8.0 * B * H * D * V + 10.0 * B * H * V)
        pv = rnd(B, delta.proj.n)
        row["vavelorn delta_step_kernel"] = _hbm(timed(lambda: ops.delta_step(delta._c, pv, st["delta"], st["ring"], seq)),
                                                 8.0 * B * H * D * V + 10.0 * B * H * V)
        rows.append(row)
        x, h = rnd(B, d, dt=torch.float32), rnd(B, d)
        experts.trace = []
        mix = experts(h)
        used = len({e for e in experts.trace[0][0].flatten().tolist() if e < E})
        experts.trace = None
        like.trace = []
        like.forward_block(h, norm.w.to(bf), 1e-6)
        used_l = len(set(like.trace[0][1].flatten().tolist()))
        like.trace = None
        one = torch.ones(d, device=dev, dtype=bf)
        by = lambda n: 2.0 * (3 * d * (n * ff + ffs) + (E + 4) * d)  # noqa: E731
        rows.append({
            "kernel": "experts, one token per sequence", "batch": B, "experts used": (used, used_l),
            "router + units + down + residual with their sum (4 launches)": _hbm(timed(lambda: ops.residual_norm(
                x, seq, bf, **{**norm.of(experts(h)), "mode": "copy"})), by(used)),
            "llama norm + router + SwiGLU + down + combine (4 launches)": _hbm(timed(lambda: like.forward_block(h, one, 1e-6)), by(used_l)),
            "router alone": round(timed(lambda: ops.moe_router(h, experts.router, experts.correction, experts.k, top, experts.groups,
                                                              experts.keep, experts._counter)) * 1e6, 1),
            "residual_norm_kernel with mixture": _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **{**norm.of(mix), "mode": "copy"})),
                                                      B * d * (10.0 + 2 * top + 2 + 2)),
            "residual_norm_kernel": _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **{**norm.of(h), "mode": "copy"})), B * d * 12.0)})
    for B, S in ((1, 4096), (8, 1024)):
        seq, n = ops.Seq(B, S, 0), B * S
        q, k, v = rnd(n, H * D), rnd(B, S, G, D), rnd(B, S, G, V)
        fl = 2.0 * B * H * (D + V) * sum(min(i + 1, W) for i in range(S))
        flc = 2.0 * B * H * (D + V) * sum(i % W + 1 for i in range(S))
        row = {"kernel": "prompt", "batch": B, "tokens": S,
               "attn_bias_prefill_kernel (window, cap, sink)": _flops(timed(lambda: ops.attn_scored(
                   q, k, v, H, G, D, V, S, 0.1, seq, cap=30.0, window=W, sinks=att.sinks)), fl, MFMA_BF16_PEAK_TFLOPS),
               "vavelorn attn_bias_prefill_kernel (chunk, cap)": _flops(timed(lambda: ops.attn_scored(
                   q, k, v, H, G, D, V, S, 0.1, seq, cap=30.0, chunk=W)), flc, MFMA_BF16_PEAK_TFLOPS)}
        big, buf, cos, sin = rnd(n, mixer.proj.n), rnd(n, mixer.width_out), *(torch.ones(S, D // 2, device=dev) for _ in range(2))
        by = 4.0 * n * (H * D + G * (D + V))
        row["qkv_headnorm_rotate_append_kernel"] = _hbm(timed(lambda: ops.qkv_headnorm_rotate_append(
            big, H, G, D, V, att.q_norm, att.k_norm, 1e-6, cos, sin, D, k, v, seq)), by)
        row["vavelorn qkv_rotate_append_kernel"] = _hbm(timed(lambda: ops.qkv_rotate_append(big, H, G, D, V, cos, sin, D, k, v, seq)), by)
        rst, ws, p, dst = ret.state(B, 4096)["retention"], ret._workspace(B, S), big[:, mixer.n_in:], buf[:, mixer.n_out:]
        fl = 5.0 * n * H * D * V  # the recurrence's own work: decay, the write, the product with q
        t = timed(lambda: ops.retention(ret._c, p, rst, ws, seq, dst))
        row["retention_prefill (3 kernels)"] = {**_flops(t, fl, FP32_MFMA_PEAK_TFLOPS),
                                                "frac_of_hbm_peak (q, k, v, gate, output)": _hbm(t, 2.0 * n * H * (2 * D + 3 * V))["frac_of_hbm_peak"]}
        st, pv, wd = delta.state(B, 4096), rnd(n, delta.proj.n), delta._workspace(B, S)
        row["vavelorn delta_prefill (3 kernels)"] = _flops(timed(lambda: ops.delta_prefill(
            delta._c, pv, None, None, st["delta"], st["ring"], wd, seq)), 7.0 * n * H * D * V, FP32_MFMA_PEAK_TFLOPS)
        x, h = rnd(n, d, dt=torch.float32), rnd(n, d)
        experts.trace = []
        mix = experts(h)
        pairs = int((experts.trace[0][0] < E).sum())
        experts.trace = None
        row["experts' share of the chosen outputs"] = round(pairs / (n * top), 3)
        row["router + sort (3 kernels)"] = _hbm(timed(lambda: ops.moe_router(
            h, experts.router, experts.correction, experts.k, top, experts.groups, experts.keep, experts._counter)), 2.0 * n * d)
        row["llama router + choice + sort (3 kernels)"] = _hbm(timed(lambda: _like_route(like, h)), 2.0 * n * d)
        row["experts (router to down)"] = _flops(timed(lambda: experts(h)), 6.0 * d * (pairs * ff + n * ffs), MFMA_BF16_PEAK_TFLOPS)
        row["llama experts (router to combine)"] = _flops(timed(lambda: like.forward_rows(h, residual=h)), 6.0 * d * n * (top * ff + ffs),
                                                          MFMA_BF16_PEAK_TFLOPS)
        row["residual_norm_kernel with mixture"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **{**norm.of(mix), "mode": "copy"})),
                                                        n * d * (10.0 + 2 * top + 2))
        row["residual_norm_kernel"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **{**norm.of(h), "mode": "copy"})), n * d * 12.0)
        rows.append(row)
    return rows


def _like_route(like, h):
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    idx, _ = like.route(h)
    n = idx.numel()
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=h.device)  # noqa: E731
    offs, pair_of, pos_of = i32(like.E + 1), i32(n), i32(n)
    check(lib().ohara_moe_sort_pairs(idx.data_ptr(), n, like.E, offs.data_ptr(), pair_of.data_ptr(), pos_of.data_ptr(), ops._stream()), "moe_sort")


def bench_fibirax(dev, sizes=("d1024", "d2048")):
    """Prefill and decode of Fibirax with random weights beside Vavelorn and Llama at the same width, depth, heads and active
    feed-forward."""
    from ohara_amd.fibirax import Fibirax, FibiraxConfig
    from ohara_amd.vavelorn import Vavelorn, VavelornConfig

    out = {}
    for name in sizes:
        cfg, vcfg = fibirax_size(name), vavelorn_size(name)
        out[name] = {"layers": len(cfg["layers"]), "width": cfg["width"], **bench_models(name, (
            ("fibirax", lambda: Fibirax(FibiraxConfig.from_dict(cfg, 4608), fibirax_state(cfg, dev), device=dev)),
            ("vavelorn", lambda: Vavelorn(VavelornConfig.from_dict(vcfg, 4608), vavelorn_state(vcfg, dev), device=dev)),
            ("llama", lambda: hybrid_llama(name, dev))), dev)}
        out[name]["kernels"] = bench_fibirax_kernels(name, dev)
        print(f"fibirax {name}: done", file=sys.stderr, flush=True)
    return out


LUDAZEN_EXPERTS = (28, 4)  # experts, used per token


def ludazen_size(name):
    """The config dict: attention with mixed heads in a window of 1024 with four kept tokens and latent attention (rank 512, a rotated
    part of 64, the same window), every second of them on the other's latents; dense feed-forwards and four of 28 experts with a
    shared one in turn, with as many active weights as a gated feed-forward of the size."""
    d, n, H, G, dh, ff = HYBRID_SIZES[name]
    experts, top = LUDAZEN_EXPERTS
    att = {"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": dh, "vdim": dh, "scale": dh ** -0.5,
                                          "mask": {"size": 1024, "keep_first": 4},
                                          "rot": {"base": 5e5, "dims": dh, "scaling": {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}}}}
    lat = {"heads": H, "dim": dh, "rot_dim": 64, "vdim": dh, "kv_rank": 512, "scale": (dh + 64) ** -0.5, "mask": {"size": 1024},
           "rot": {"base": 5e5, "dims": 64}}
    dense = {"kind": "dense", "ff": 3 * ff // 2}
    moe = {"kind": "moe", "router": {"experts": experts, "top": top}, "expert": {"ff": ff // 8}, "shared": {"ff": ff // 2}}
    layers = []
    for i in range(0, n, 4):
        layers += [{**att, "mlp": dense}, {"type": "latent_attention", "mixer": lat, "mlp": moe},
                   {"type": "latent_attention", "mixer": {**lat, "kv_from": i + 1}, "mlp": dense}, {**att, "mlp": moe}]
    return {"width": d, "vocab": 32000, "norm": {"eps": 1e-6}, "layers": layers}


def ludazen_state(cfg, dev, seed=5):
    """Random weights: matrices N(0, 1/columns), unit norms and temperatures."""
    g = torch.Generator(device=dev).manual_seed(seed)
    n = lambda *shape, s=1.0: (torch.randn(*shape, generator=g, device=dev) * s).to(torch.bfloat16)  # noqa: E731
    lin = lambda o, i: n(o, i, s=i ** -0.5)  # noqa: E731
    one = lambda k: torch.ones(k, device=dev, dtype=torch.bfloat16)  # noqa: E731
    d = cfg["width"]
    st = {"embed": n(cfg["vocab"], d), "head": lin(cfg["vocab"], d), "final.norm": one(d)}
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        H, D, V, q = m["heads"], m["dim"], m["vdim"], p + "mix."
        st.update({p + "norm1": one(d), p + "norm2": one(d), q + "o": lin(d, H * V)})
        if layer["type"] == "attention":
            G = m["kv_heads"]
            st.update({q + "q": lin(H * D, d), q + "k": lin(G * D, d), q + "v": lin(G * V, d), q + "temp": one(H), q + "talk": lin(H, H)})
        else:
            r, e = m["kv_rank"], m["rot_dim"]
            st.update({q + "q": lin(H * (D + e), d), q + "uk": lin(H * D, r), q + "uv": lin(H * V, r)})
            if "kv_from" not in m:
                st.update({q + "dkv": lin(r + e, d), q + "dkv.norm": one(r)})
        q = p + "mlp."
        if mlp["kind"] == "dense":
            st.update({q + "up": lin(mlp["ff"], d), q + "up.b": n(mlp["ff"], s=0.1), q + "down": lin(d, mlp["ff"]), q + "down.b": n(d, s=0.1),
                       q + "act": n(2)})
            continue
        st[q + "router"] = lin(mlp["router"]["experts"], d)
        for name, ff in [(f"e{e}", mlp["expert"]["ff"]) for e in range(mlp["router"]["experts"])] + [("shared", mlp["shared"]["ff"])]:
            st.update({f"{q}{name}.gate": lin(ff, d), f"{q}{name}.up": lin(ff, d), f"{q}{name}.down": lin(d, ff)})
    return st


def bench_ludazen_kernels(name, dev):
    """The design's own kernels at one layer's sizes, each beside the like kernel of Vavelorn or Fibirax."""
    from ohara_amd import ops
    from ohara_amd._lib import ROUTER_PLAIN, ROUTER_SIGMOID
    from ohara_amd.fibirax import Fibirax, FibiraxConfig
    from ohara_amd.hybrid import added
    from ohara_amd.ludazen import Ludazen, LudazenConfig
    from ohara_amd.vavelorn import Vavelorn, VavelornConfig

    bf, cfg, vcfg, fcfg = torch.bfloat16, ludazen_size(name), vavelorn_size(name), fibirax_size(name)
    cfg, fcfg = {**cfg, "layers": cfg["layers"][:2]}, {**fcfg, "layers": fcfg["layers"][:1]}
    model = Ludazen(LudazenConfig.from_dict(cfg, 4096), ludazen_state(cfg, dev), device=dev)
    vlat = _sole_layers(Vavelorn, VavelornConfig.from_dict, vavelorn_state(vcfg, dev), vcfg, ("latent_attention",), dev).layers[0]["mixer"]
    fib = Fibirax(FibiraxConfig.from_dict(fcfg, 4096), fibirax_state(fcfg, dev), device=dev).layers[0]
    fexp, fnorm = fib["mlp"], fib["norm2"]
    att, lat, mlp, experts, norm = *(b["mixer"] for b in model.layers), model.layers[0]["mlp"], model.layers[1]["mlp"], model.layers[0]["norm1"]
    H, G, D, V, d, W, R, E = att.heads, att.kv_heads, att.dim, att.vdim, cfg["width"], att.window, lat.rank, lat.rot_dim
    C, K, ff = lat.row, att.keep_first, mlp.up.n
    rnd = lambda *shape, dt=bf: torch.randn(*shape, device=dev).to(dt)  # noqa: E731
    rows = []

    def timed(fn, n=8):  # n calls per graph: what a single-launch graph costs to start would swamp the small kernels
        return graph_time(lambda: [fn() for _ in range(n)], iters=20) / n

    for B, L in ((1, 4096), (8, 4096), (32, 2048)):
        seq, short = ops.Seq(B, 1, L - 1), ops.Seq(B, 1, W - 1)
        q, k, v = rnd(B, H * D), rnd(B, L, G, D), rnd(B, L, G, V)
        nm, wm = att._split(B, L)
        nf = max(1, min(1024 // (B * G * -(-(H // G) // 4)), W // 128, 64))
        wf = ops.attn_bias_workspace(B, H, V, nf, dev) if nf > 1 else None
        c, cl, ql, qv = rnd(B, L, C), rnd(B, W, R), rnd(B, H * C), rnd(B, H * R)
        nl, wl = lat._split(B, L)
        nv, wv = vlat._split(B, W)
        by = 2.0 * G * (D + V) * B * W
        rows.append({
            "kernel": "decode attention", "batch": B, "context": L, "window": W,
            "mixed scores + values (window, kept)": _hbm(timed(lambda: ops.attn_mixed(
                q, k, v, H, G, D, V, 0.1, att.talk, seq, temp=att.temp, window=W, keep=K, n_split=nm, workspace=wm)), by),
            "attn_bias_kernel (window), Fibirax": _hbm(timed(lambda: ops.attn_scored(
                q, k, v, H, G, D, V, L, 0.1, seq, window=W, n_split=nf, workspace=wf)), by),
            "attn_latent_kernel + merge (window, key part)": _hbm(timed(lambda: ops.attn_latent(ql, c, H, R, 0.1, seq, nl, wl, window=W)),
                                                                  2.0 * C * B * W),
            "attn_latent_kernel + merge, Vavelorn": _hbm(timed(lambda: ops.attn_latent(qv, cl, H, R, 0.1, short, nv, wv)), 2.0 * R * B * W)})
        p, cos, sin = rnd(B, max(lat.proj.n, vlat.proj.n)), *(torch.ones(L, E // 2, device=dev) for _ in range(2))
        h, x, a = rnd(B, d), rnd(B, d, dt=torch.float32), rnd(B, ff)
        plain_up, plain_down = ops.pack_linear(rnd(ff, d)), ops.pack_linear(rnd(d, ff))
        row = {"kernel": "one token", "batch": B}
        row["latent_rotary_front_kernel"] = _hbm(timed(lambda: ops.latent_rotary_front(
            p, H, D, cos, sin, ql[:, R:], C, seq, cache=c, off_c=lat.n_q, off_r=lat.n_q + R, rank=R, cn=lat.kv_norm, eps=1e-6)),
            4.0 * B * (H * E + C))
        row["latent_front_kernel, Vavelorn"] = _hbm(timed(lambda: ops.latent_front(
            p, vlat.q_rank, vlat.off_c, R, vlat.q_norm, vlat.kv_norm, 1e-5, cl, ops.Seq(B, 1, W - 1))), 4.0 * B * (vlat.q_rank + R))
        wby = 2.0 * ff * d
        row["gemm_xielu"] = _hbm(timed(lambda: ops.gemm_xielu(h, mlp.up.w, mlp.up.bias, mlp.above, mlp.below)), wby)
        row["gemm_skinny, same weights"] = _hbm(timed(lambda: ops.gemm_skinny(h, plain_up)), wby)
        row["linear_bias (down)"] = _hbm(timed(lambda: mlp.down(a)), wby)
        row["gemm_skinny, same weights (down)"] = _hbm(timed(lambda: ops.gemm_skinny(a, plain_down)), wby)
        row["head_linear_kernel (keys, heads apart)"] = _hbm(timed(lambda: ops.head_linear(
            p, lat.k_absorb, R, out=ql, x_heads=lat.dq + lat.dr, out_heads=C)), 2.0 * H * R * D)
        row["head_linear_kernel (keys), Vavelorn"] = _hbm(timed(lambda: ops.head_linear(q, vlat.k_absorb, R)), 2.0 * H * R * D)
        row["residual_norm_kernel (sum)"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **added(h), **norm.out())), B * d * 12.0)
        row["residual_norm_kernel (two norms)"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **norm.of(h), mode="norm", norm2_w=norm.w)),
                                                       B * d * 12.0)
        for label, m, nrm, total in (("", experts, None, LUDAZEN_EXPERTS[0]), (", Fibirax", fexp, fnorm, sum(FIBIRAX_EXPERTS[:2]))):
            m.trace = []
            m(h)
            used = len({e for e in m.trace[0][0].flatten().tolist() if e < m.experts})
            m.trace = None
            row[f"experts with their sum{label} ({used} used)"] = _hbm(
                timed(lambda: ops.residual_norm(x, seq, bf, **({**added(m(h)), **norm.out()} if nrm is None else {**nrm.of(m(h)), "mode": "copy"}))),  # noqa: B023
                2.0 * (3 * d * (used * m.ff + m.shared.ff) + (total + 4) * d))
        rows.append(row)
    for B, S in ((1, 4096), (8, 1024)):
        seq, n = ops.Seq(B, S, 0), B * S
        q, k, v = rnd(n, H * D), rnd(B, S, G, D), rnd(B, S, G, V)
        pairs = B * sum(min(i + 1, W) for i in range(S))
        fl = 2.0 * H * (D + V) * pairs
        kv, part, ql = rnd(n, H * (D + V)), rnd(n, E), rnd(n, H * (D + E))
        row = {"kernel": "prompt", "batch": B, "tokens": S}
        row["mixed_prefill_kernel + packing"] = _flops(timed(lambda: ops.attn_mixed(
            q, k, v, H, G, D, V, 0.1, att.talk, seq, temp=att.temp, window=W, keep=K)), fl + 2.0 * H * H * pairs, MFMA_BF16_PEAK_TFLOPS)
        row["attn_bias_prefill_kernel (window), Fibirax"] = _flops(timed(lambda: ops.attn_scored(q, k, v, H, G, D, V, S, 0.1, seq, window=W)), fl,
                                                                   MFMA_BF16_PEAK_TFLOPS)
        row["latent: attn_bias_prefill_kernel (window, shared key part)"] = _flops(timed(lambda: ops.attn_scored(
            ql, kv, kv[:, H * D:], H, H, D + E, V, S, 0.1, seq, window=W, ld_k=kv.stride(0), ld_v=kv.stride(0), k_shared=part, ld_shared=E, d_shared=E)),
            2.0 * H * (D + E + V) * pairs, MFMA_BF16_PEAK_TFLOPS)
        row["latent: attn_bias_prefill_kernel (window), Vavelorn"] = _flops(timed(lambda: ops.attn_scored(
            q, kv, kv[:, H * D:], H, H, D, V, S, 0.1, seq, window=W, ld_k=kv.stride(0), ld_v=kv.stride(0))), fl, MFMA_BF16_PEAK_TFLOPS)
        p, cos, sin, c, cl = rnd(n, max(lat.proj.n, vlat.proj.n)), *(torch.ones(S, E // 2, device=dev) for _ in range(2)), rnd(B, S, C), rnd(B, S, R)
        row["latent_rotary_front_kernel"] = _hbm(timed(lambda: ops.latent_rotary_front(
            p, H, D, cos, sin, p[:, D:], D + E, seq, cache=c, off_c=lat.n_q, off_r=lat.n_q + R, rank=R, cn=lat.kv_norm, eps=1e-6, compact=True)),
            2.0 * n * (2 * H * E + 3 * C))
        row["latent_front_kernel, Vavelorn"] = _hbm(timed(lambda: ops.latent_front(
            p, vlat.q_rank, vlat.off_c, R, vlat.q_norm, vlat.kv_norm, 1e-5, cl, seq, True)), 2.0 * n * (2 * vlat.q_rank + 3 * R))
        h, x = rnd(n, d), rnd(n, d, dt=torch.float32)
        plain = ops.pack_linear(rnd(ff, d))
        row["gemm_xielu"] = _flops(timed(lambda: ops.gemm_xielu(h, mlp.up.w, mlp.up.bias, mlp.above, mlp.below)), 2.0 * n * d * ff, MFMA_BF16_PEAK_TFLOPS)
        row["gemm, same weights"] = _flops(timed(lambda: ops.gemm_skinny(h, plain)), 2.0 * n * d * ff, MFMA_BF16_PEAK_TFLOPS)
        row["router + sort (3 kernels)"] = _hbm(timed(lambda: ops.moe_router(
            h, experts.router, None, experts.k, experts.top, 1, 1, experts._counter, ROUTER_SIGMOID | ROUTER_PLAIN)), 2.0 * n * d)
        row["router + sort, Fibirax"] = _hbm(timed(lambda: ops.moe_router(
            h, fexp.router, fexp.correction, fexp.k, fexp.top, fexp.groups, fexp.keep, fexp._counter)), 2.0 * n * d)
        for label, m in (("", experts), (", Fibirax", fexp)):
            m.trace = []
            m(h)
            used = int((m.trace[0][0] < m.experts).sum())
            m.trace = None
            row["experts (router to down)" + label] = _flops(timed(lambda: m(h)), 6.0 * d * (used * m.ff + n * m.shared.ff), MFMA_BF16_PEAK_TFLOPS)  # noqa: B023
        row["residual_norm_kernel (sum)"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **added(h), **norm.out())), n * d * 12.0)
        row["residual_norm_kernel (two norms)"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **norm.of(h), mode="norm", norm2_w=norm.w)),
                                                       n * d * 12.0)
        mix, fmix = experts(h), fexp(h)
        row["residual_norm_kernel (sum of a mixture)"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **added(mix), **norm.out())),
                                                              n * d * (10.0 + 2 * experts.top + 2))
        row["residual_norm_kernel (norm of a mixture), Fibirax"] = _hbm(timed(lambda: ops.residual_norm(x, seq, bf, **{**fnorm.of(fmix), "mode": "copy"})),
                                                                        n * d * (10.0 + 2 * fexp.top + 2))
        rows.append(row)
    return rows


def bench_ludazen(dev, sizes=("d1024", "d2048")):
    """Prefill and decode of Ludazen with random weights beside Fibirax, Vavelorn and Llama at the same width, depth, heads and active
    feed-forward."""
    from ohara_amd.fibirax import Fibirax, FibiraxConfig
    from ohara_amd.ludazen import Ludazen, LudazenConfig
    from ohara_amd.vavelorn import Vavelorn, VavelornConfig

    out = {}
    for name in sizes:
        cfg, vcfg, fcfg = ludazen_size(name), vavelorn_size(name), fibirax_size(name)
        out[name] = {"layers": len(cfg["layers"]), "width": cfg["width"], **bench_models(name, (
            ("ludazen", lambda: Ludazen(LudazenConfig.from_dict(cfg, 4608), ludazen_state(cfg, dev), device=dev)),
            ("fibirax", lambda: Fibirax(FibiraxConfig.from_dict(fcfg, 4608), fibirax_state(fcfg, dev), device=dev)),
            ("vavelorn", lambda: Vavelorn(VavelornConfig.from_dict(vcfg, 4608), vavelorn_state(vcfg, dev), device=dev)),
            ("llama", lambda: hybrid_llama(name, dev))), dev)}
        out[name]["kernels"] = bench_ludazen_kernels(name, dev)
        print(f"ludazen {name}: done", file=sys.stderr, flush=True)
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=256)
    ap.add_argument("--warmup", type=int, default=16)
    ap.add_argument("--prompt", type=int, default=1024)
    ap.add_argument("--batches", type=str, default="1,8,32,64")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-extended", action="store_true",
                    help="skip the per-kernel figures of the other configurations (attention microbench, "
                         "prefill on MFMA, BitNet and MoE decode)")
    ap.add_argument("--pmc-calibration", action="store_true",
                    help="also run three 1 GiB device-to-device copies (a kernel of known traffic to scale "
                         "FETCH_SIZE / WRITE_SIZE counters against)")
    ap.add_argument("--timeline-batch", type=int, default=1, help="sequences of the --phase-timeline run (1 to 8)")
    ap.add_argument("--timeline-int8", action="store_true", help="the --phase-timeline run over an int8 KV cache")
    ap.add_argument("--phase-timeline", action="store_true",
                    help="print the per-phase timeline of the persistent decode kernel at batch 1 and exit")
    ap.add_argument("--bitnet-phase-timeline", type=int, default=0, metavar="B",
                    help="print the per-phase timeline of the single-launch BitNet decode step at batch B and exit")
    ap.add_argument("--bitnet-only", type=str, default="", metavar="BATCHES",
                    help="run the BitNet ternary decode figures alone at these batch sizes (e.g. 1,8) and exit "
                         "(profiling workload)")
    ap.add_argument("--moe-only", action="store_true",
                    help="run the MoE decode figure alone and exit (profiling workload)")
    ap.add_argument("--prefill-only", action="store_true",
                    help="run the d12 prefill figures (tiled MFMA GEMMs, prefill attention) alone and exit")
    ap.add_argument("--attention-only", action="store_true",
                    help="run the GQA decode-attention figures (bf16 and int8 cache) alone and exit")
    ap.add_argument("--povazen-only", type=str, nargs="?", const="d1024,d2048", default="", metavar="SIZES",
                    help="run the Povazen prefill, decode and kernel figures beside Llama at equal sizes alone and exit")
    ap.add_argument("--vavelorn-only", type=str, nargs="?", const="d1024,d2048", default="", metavar="SIZES",
                    help="run the Vavelorn prefill, decode and kernel figures beside Povazen and Llama at equal sizes alone and exit")
    ap.add_argument("--fibirax-only", type=str, nargs="?", const="d1024,d2048", default="", metavar="SIZES",
                    help="run the Fibirax prefill, decode and kernel figures beside Vavelorn and Llama at equal sizes alone and exit")
    ap.add_argument("--ludazen-only", type=str, nargs="?", const="d1024,d2048", default="", metavar="SIZES",
                    help="run the Ludazen prefill, decode and kernel figures beside Fibirax, Vavelorn and Llama at equal sizes alone and exit")
    ap.add_argument("--phi-decode-only", type=int, default=0, metavar="B",
                    help="run 12 eager Phi-2 decode steps of B sequences at context 1024 and exit (profiling workload)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this build runs on ONE MI355X (no sharding, no collectives); --gpus must be 1",
              file=sys.stderr)
        sys.exit(2)
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(1)

    from ohara_amd.llama import Llama

    dev = torch.device("cuda:0")
    if args.pmc_calibration:
        src = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    if args.povazen_only:
        print(json.dumps(bench_povazen(dev, tuple(args.povazen_only.split(","))), indent=1))
        return
    if args.vavelorn_only:
        print(json.dumps(bench_vavelorn(dev, tuple(args.vavelorn_only.split(","))), indent=1))
        return
    if args.fibirax_only:
        print(json.dumps(bench_fibirax(dev, tuple(args.fibirax_only.split(","))), indent=1))
        return
    if args.ludazen_only:
        print(json.dumps(bench_ludazen(dev, tuple(args.ludazen_only.split(","))), indent=1))
        return
    if args.phi_decode_only:
        print(json.dumps(phi_decode_only(dev, args.phi_decode_only)))
        return
    if args.bitnet_phase_timeline:
        print(json.dumps(bitnet_phase_timeline(dev, args.bitnet_phase_timeline), indent=1))
        return
    if args.moe_only:
        print(json.dumps(bench_moe(dev), indent=1))
        return
    if args.attention_only:
        print(json.dumps(bench_attention_microbench(dev), indent=1))
        return
    if args.bitnet_only:
        print(json.dumps(bench_bitnet(dev, tuple(int(b) for b in args.bitnet_only.split(","))), indent=1))
        return
    if args.phase_timeline:
        print(json.dumps(phase_timeline(dev, args.prompt, batch=args.timeline_batch, int8=args.timeline_int8), indent=1))
        return
    cfg, st = d12_state(dev)
    model = Llama(cfg, st, device=dev)
    del st
    if args.prefill_only:
        print(json.dumps(bench_prefill(model, cfg, dev), indent=1))
        return
    batches = [int(b) for b in args.batches.split(",") if b]
    if 1 not in batches:
        batches = [1] + batches
    results = {}
    roof = None
    lm_index = 1 + 5 * cfg.num_hidden_layers
    for b in batches:
        dt, l_mean, sess = time_decode(model, b, args.prompt, args.warmup, args.steps)
        ms = dt / args.steps * 1e3
        by = step_bytes(cfg, b, l_mean)
        results[b] = {"tokens_per_s": round(b * args.steps / dt, 1), "ms_per_step": round(ms, 4),
                      "step_bytes": int(by), "step_GBs": round(by / (dt / args.steps) / 1e9, 1),
                      "step_frac_of_hbm_peak": round(by / (dt / args.steps) / 1e9 / HBM_PEAK_GBS, 4)}
        results[b]["launch"] = "one persistent kernel per step" if sess.persistent else "63 kernels per step"
        if b == 1:
            # the dominant kernel, timed with HIP events on the launch stream inside real
            # decode steps of a fresh session that continues from the same prompt length
            n_prof = 64
            sess2 = model.session(1, args.warmup + n_prof + 8)
            sess2.prefill(torch.randint(0, cfg.vocab_size, (1, args.prompt)).to(dev))
            for _ in range(args.warmup):
                sess2.step()
            torch.cuda.synchronize()
            t_k = time_kernel_in_situ(sess2, lm_index, n_prof)
            sess2.check_error()
            if sess2.persistent:
                kb = step_bytes(cfg, 1, args.prompt + args.warmup + (n_prof + 1) / 2.0)
                kname = "decode_mega_kernel<128,1,1,false,false> (batch-1 polled build; whole decode step: 12 layers + vocabulary projection + selection)"
            else:
                kb = lm_head_bytes(cfg, 1)
                kname = "wide_kernel<1,true,STORE> (final norm + vocabulary projection 65536x768)"
            roof = {"kernel": kname, "bound": "hbm", "achieved": round(kb / t_k / 1e9, 1), "peak": HBM_PEAK_GBS,
                    "unit": "GB/s", "frac": round(kb / t_k / 1e9 / HBM_PEAK_GBS, 4),
                    "traffic": PMC_TRAFFIC_BYTES.get(("persistent" if sess2.persistent else "chain", 1, args.prompt)),
                    "traffic_source": "constant carried in bench.py from two rocprofv3 --pmc runs (FETCH_SIZE, WRITE_SIZE) "
                                      "summarised in profiles/decode_mega_kernel_d12_batch1_pmc.txt; not measured by this run",
                    "bytes_per_launch": int(kb), "avg_launch_us": round(t_k * 1e6, 2)}
        del sess
        torch.cuda.empty_cache()

    # the same decode at batch 1 with temperature 0.8 / top-k 50 / top-p 0.9 sampling from a
    # pre-drawn uniform tensor (forward + fused sampler per step, replayed from one graph)
    from ohara_amd.sampling import SamplingConfig

    dt, _, sess = time_decode(model, 1, args.prompt, args.warmup, args.steps,
                              sampling=SamplingConfig(temperature=0.8, top_k=50, top_p=0.9))
    results["1_sampled"] = {"tokens_per_s": round(args.steps / dt, 1), "ms_per_step": round(dt / args.steps * 1e3, 4),
                            "sampling": "temperature 0.8, top-k 50, top-p 0.9, seeded uniform draws",
                            "launch": "persistent kernel + sampler kernel per step"}
    del sess
    torch.cuda.empty_cache()
    # the int8 KV cache (codes + a scale and a minimum per head row) through the same single launch
    for b in (1, 8):
        dt, l_mean, sess = time_decode(model, b, args.prompt, args.warmup, args.steps, int8=True)
        by = step_bytes(cfg, b, l_mean, int8=True)
        results[f"{b}_int8_cache"] = {
            "tokens_per_s": round(b * args.steps / dt, 1), "ms_per_step": round(dt / args.steps * 1e3, 4),
            "step_bytes": int(by), "step_frac_of_hbm_peak": round(by / (dt / args.steps) / 1e9 / HBM_PEAK_GBS, 4),
            "launch": "one persistent kernel per step" if sess.persistent else "kernel chain"}
        del sess
        torch.cuda.empty_cache()
    r1 = results[1]
    out = {
        "metric": "decode tokens/s at batch 1 & 32 (d12 Llama, 4k ctx) + % of HBM roofline",
        "value": r1["tokens_per_s"], "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": r1["ms_per_step"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": f"d12 Llama bf16 greedy decode, batch 1, prompt {args.prompt}, KV cache 4096 "
                               f"(the configuration the metric is quoted on)", "batch": 1, "prompt_len": args.prompt,
                   "context_capacity": 4096, "launch": r1["launch"] + ", HIP graph replay"},
        "also": {f"batch{b}": r for b, r in results.items()},
        "roofline": roof,
    }
    out["also"]["chat_engine_batch1"] = bench_chat_engine(model, cfg, dev, args.prompt, args.steps, args.warmup)
    if not args.no_extended:
        out["also"]["continuous_batch32"] = bench_continuous(model, cfg, dev)
        out["kernels"] = {"prefill_d12": bench_prefill(model, cfg, dev)}
        del model
        torch.cuda.empty_cache()
        out["kernels"]["decode_attention_gqa_32q_8kv_128"] = bench_attention_microbench(dev)
        out["kernels"]["bitnet_decode"] = bench_bitnet(dev)
        out["kernels"]["moe_decode"] = bench_moe(dev)
        out["kernels"]["phi2_decode"] = bench_phi(dev)
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline()
    print(json.dumps(out))


if __name__ == "__main__":
    main()
