"""The calls whose speed is measured, as a serving program makes them.

Every pass is one call of the C ABI (include/pa_mi355x.h) the way a plugin's Compute body makes it:
device tensors, the node's attributes and the host copies of the int32 metadata in descriptors that
the program keeps, a workspace sized once by the library, and the current stream.  The calls are

  paged    pa_paged_attention: RMSNorm / RoPE / append of the new tokens, then attention over the
           pages; decode batches, chunked prefill, both in one batch, and the LATENT layout
  gqa      pa_group_query_attention: contiguous past / present caches, decode and first prompts
  append   pa_reshape_and_cache alone

A case holds sizes and options only.  `layout` seeds the ragged lengths (so work() can count them);
the seed of prepare() makes the tensors and the order of the pages.
"""
from __future__ import annotations

import ctypes as C
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "onnxruntime-ep-mlx_amd"))

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ELEM = {"bf16": 2.0, "f16": 2.0, "f32": 4.0}
CODED = {"fp8": 1.0, "int8": 1.0, "int4": 0.5}  # bytes per element of a byte-coded cache


def _paged(name=None, **kw):
    # steps: sequences with `step` new tokens each, over `past_min`..`past_max` cached ones;
    # chunks: sequences with chunk_min..chunk_max new tokens over chunk_past_min..chunk_past_max.
    c = dict(call="paged", dtype="bf16", cache="same", heads=32, kv=8, head=128, latent=False,
             block=16, steps=0, step=1, past_min=0, past_max=0, chunks=0, chunk_min=0, chunk_max=0,
             chunk_past_min=0, chunk_past_max=0, rotary=0, theta=500000.0, window=-1, sink=False,
             softcap=0.0, norm=False, layout=3)
    c.update(kw)
    return c if name is None else dict(name=name, **c)


def _gqa(name=None, **kw):
    # seq new tokens per sequence; capacity 0: a first prompt without a past, new presents
    # (lengths seq_min..seq, right-padded); else shared presents of `capacity` rows.
    c = dict(call="gqa", dtype="bf16", cache="same", heads=32, kv=8, head=128, batch=1, seq=1,
             seq_min=0, past_min=0, past_max=0, capacity=0, rotary=0, theta=500000.0, window=-1,
             sink=False, softcap=0.0, layout=3)
    c.update(kw)
    return c if name is None else dict(name=name, **c)


def _append(name=None, **kw):
    c = dict(call="append", dtype="f16", cache="same", kv=8, head=128, block=16, batch=32,
             new_min=1, new_max=1, past_min=128, past_max=2048, distinct=False, layout=2)
    c.update(kw)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # The smallest call: one token of one sequence against a short contiguous past in fp32
        # (a small on-device model's decode); launches and latency are all of it.
        _gqa("gqa_f32_one_token", dtype="f32", heads=8, kv=2, head=64, batch=1, seq=1, past_min=128,
             past_max=128, capacity=192),
        # The KV append alone, for an engine that schedules append and attention itself.
        _append("append_f16_32"),
        # One interactive user of a long session: head 256, QK norm, partial rotary, 256-row pages,
        # 16K context; the chip has one sequence and four kv-heads to split.
        _paged("decode_one_16k", dtype="f16", heads=24, kv=4, head=256, block=256, steps=1,
               past_min=16383, past_max=16383, rotary=64, theta=10000000.0, norm=True),
        # A lightly loaded server: a few conversations that have just begun.
        _paged("decode_small_batch", steps=8, past_min=60, past_max=1500, rotary=128),
        # A loaded server: the Llama-3-8B-shaped decode step.
        _paged("decode_batch_64", steps=64, past_min=511, past_max=8191, rotary=128),
        # Long documents over fp8 pages.
        _paged("decode_fp8_32k", cache="fp8", heads=64, kv=8, steps=16, past_min=32767,
               past_max=32767),
        # GroupQueryAttention with an int4 present updated in place, a loaded server's step.
        _gqa("gqa_decode_int4", cache="int4", batch=64, seq=1, past_min=511, past_max=8190,
             capacity=8192, rotary=128),
        # Chunked prefill, Qwen2.5-7B-shaped: eight 512-token chunks over cached contexts.
        _paged("prefill_chunks", heads=28, kv=4, chunks=8, chunk_min=512, chunk_max=512,
               chunk_past_max=4096, layout=4),
        # Continuous batching: most sequences decode while new requests prefill in the same call.
        _paged("mixed_batch", steps=48, past_min=100, past_max=6000, chunks=3, chunk_min=100,
               chunk_max=600, chunk_past_max=2048, rotary=128, layout=5),
        # Prompts on a sliding-window layer with attention sinks, head 64.
        _paged("prefill_window_sink", dtype="f16", heads=64, kv=8, head=64, chunks=4,
               chunk_min=301, chunk_max=1500, chunk_past_max=1000, rotary=64, theta=150000.0,
               window=128, sink=True, layout=6),
        # A first prompt through GroupQueryAttention: no past, presents returned.
        _gqa("gqa_prompt_1023", dtype="f16", batch=2, seq=1023, seq_min=1023, rotary=128),
        # MLA decode with absorbed projections: 128 query heads over one 576-wide latent row.
        _paged("mla_decode_128", heads=128, kv=1, head=576, latent=True, steps=64, past_min=511,
               past_max=8191, rotary=64, theta=10000.0),
    ]


# ------------------------------------------------------------------------------------- drawing

def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


MOST_BYTES, MOST_FLOPS = 1.0e9, 7.0e10


def _within(case):
    w = work(case)
    return w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS


def draw(rng):
    while True:
        kind = rng.choices(("decode", "prefill", "gqa", "latent", "append"),
                           (0.3, 0.3, 0.2, 0.12, 0.08))[0]
        layout = rng.randrange(1 << 20)
        if kind == "append":
            case = _append(dtype=rng.choice(("f16", "bf16")),
                           cache=rng.choice(("same", "same", "fp8", "int8")),
                           kv=rng.choice((4, 8)), head=rng.choice((64, 128, 256)),
                           block=rng.choice((16, 32, 256)), batch=_logint(rng, 1, 64),
                           new_min=1, new_max=_logint(rng, 1, 300), past_min=0, past_max=2048,
                           distinct=rng.random() < 0.5, layout=layout)
        elif kind == "latent":
            longest = _logint(rng, 200, 8191)
            case = _paged(dtype=rng.choice(("bf16", "f16")), heads=rng.choice((16, 32, 64, 128)),
                          kv=1, head=576, latent=True, block=rng.choice((16, 32, 64)),
                          steps=_logint(rng, 1, 64), step=rng.choice((1, 1, 2)),
                          past_min=longest // 16, past_max=longest, rotary=64, theta=10000.0,
                          layout=layout)
        elif kind == "gqa":
            heads, kv, head = rng.choice(((32, 8, 128), (28, 4, 128), (64, 8, 64), (24, 4, 256)))
            pick = rng.random()
            if pick < 0.1:
                longest = _logint(rng, 64, 2048)
                case = _gqa(dtype="f32", heads=8, kv=2, head=64, batch=_logint(rng, 1, 8),
                            past_min=longest // 2, past_max=longest, capacity=longest + 64,
                            layout=layout)
            elif pick < 0.6:
                longest = _logint(rng, 64, 8190)
                case = _gqa(dtype=rng.choice(("bf16", "f16")),
                            cache=rng.choice(("same", "same", "int8", "int4"))
                            if head in (64, 128) else "same",
                            heads=heads, kv=kv, head=head, batch=_logint(rng, 1, 64), seq=1,
                            past_min=longest // 16, past_max=longest, capacity=longest + 2,
                            rotary=head, window=rng.choice((-1, -1, -1, 1024)), layout=layout)
            else:
                seq = _logint(rng, 20, 2048)
                case = _gqa(dtype=rng.choice(("bf16", "f16")), heads=heads, kv=kv, head=head,
                            batch=_logint(rng, 1, 8), seq=seq,
                            seq_min=seq if rng.random() < 0.5 else max(1, seq // 3), rotary=head,
                            softcap=rng.choice((0.0, 0.0, 0.0, 50.0)), layout=layout)
        else:
            heads, kv, head = rng.choice(((32, 8, 128), (28, 4, 128), (64, 8, 128), (64, 8, 64),
                                          (24, 4, 256)))
            case = _paged(dtype=rng.choice(("bf16", "bf16", "f16")),
                          cache=rng.choice(("same", "same", "same", "fp8", "int8"))
                          if head in (64, 128) else "same",
                          heads=heads, kv=kv, head=head, block=rng.choice((16, 16, 32, 256)),
                          rotary=rng.choice((head, head, 0)), norm=rng.random() < 0.2,
                          window=rng.choice((-1, -1, -1, 128, 1024)), sink=rng.random() < 0.15,
                          softcap=rng.choice((0.0, 0.0, 0.0, 0.0, 50.0)), layout=layout)
            if kind == "decode":
                longest = _logint(rng, 64, 32000)
                case.update(steps=_logint(rng, 1, 64), step=rng.choice((1, 1, 1, 2)),
                            past_min=longest // 16, past_max=longest)
            else:
                longest = _logint(rng, 20, 2048)
                past = rng.choice((0, _logint(rng, 16, 4096)))
                case.update(chunks=_logint(rng, 1, 8), chunk_min=max(1, longest // 4),
                            chunk_max=longest, chunk_past_max=past)
                if rng.random() < 0.4:
                    longest = _logint(rng, 64, 8000)
                    case.update(steps=_logint(rng, 1, 48), past_min=longest // 16,
                                past_max=longest)
        if _within(case):
            return case


# ------------------------------------------------------------------------------ lengths and work

def _lengths(case):
    """[(new tokens, past tokens)] of every sequence, in batch order."""
    rng = random.Random(case["layout"])
    if case["call"] == "append":
        return [(rng.randint(case["new_min"], case["new_max"]),
                 rng.randint(case["past_min"], case["past_max"])) for _ in range(case["batch"])]
    if case["call"] == "gqa":
        if case["capacity"] == 0:
            lens = [rng.randint(case["seq_min"], case["seq"]) for _ in range(case["batch"])]
            lens[0] = case["seq"]
            return [(n, 0) for n in lens]
        return [(case["seq"], rng.randint(case["past_min"], case["past_max"]))
                for _ in range(case["batch"])]
    seqs = [(case["step"], rng.randint(case["past_min"], case["past_max"]))
            for _ in range(case["steps"])]
    seqs += [(rng.randint(case["chunk_min"], case["chunk_max"]),
              rng.randint(case["chunk_past_min"], case["chunk_past_max"]))
             for _ in range(case["chunks"])]
    rng.shuffle(seqs)
    return seqs


def _v_head(case):
    return 512 if case.get("latent") else case["head"]


def work(case):
    es = ELEM[case["dtype"]]
    cb = CODED.get(case["cache"], es)
    lens = _lengths(case)
    kv, d = case["kv"], case["head"]
    sides = 1 if case.get("latent") else 2
    row = kv * d * sides  # elements of one position's key and value rows
    if case["call"] == "append":
        return {"bytes": sum(n for n, _ in lens) * row * (es + cb), "flops": 0.0}
    H, vd, win = case["heads"], _v_head(case), case["window"]
    prompt = case["call"] == "gqa" and case["capacity"] == 0
    nbytes = pairs = 0.0
    for n, past in lens:
        first = max(0, past - win + 1) if win > 0 else 0
        nbytes += (past - first) * row * cb + n * row * (es + cb)
        rows = case["seq"] if prompt else n  # a right-padded prompt computes its padding rows too
        nbytes += rows * H * (d + vd) * es
        i = np.arange(rows, dtype=np.float64)
        hi = np.minimum(past + i + 1, past + n)
        lo = np.maximum(0, np.minimum(past + i, past + n - 1) - win + 1) if win > 0 else 0
        pairs += float(np.sum(hi - lo))
    if case["cache"] in ("fp8",):
        nbytes += sum(-(-(n + p) // case["block"]) for n, p in lens) * kv * 4 * sides
    return {"bytes": nbytes, "flops": 2.0 * H * (d + vd) * pairs}


def tolerance(case):
    if case["call"] == "append":
        return "exact"
    # Outputs are rounded once to the activation type; the attention is summed in 32 bits.
    rel = {"f32": 4e-6, "f16": 1.6e-3, "bf16": 8e-3}[case["dtype"]]
    return {"rel": rel, "max": {"f32": 1e-4, "f16": 0.02, "bf16": 0.08}[case["dtype"]]}


# --------------------------------------------------------------------------------------- inputs

def _quantise(x, scale, cache, reciprocal=False):
    """Codes of rows x [..., head] under `scale` (broadcastable), as the cache stores them."""
    if cache == "fp8":
        return (x.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
    y = x.float() * (1.0 / scale) if reciprocal else x.float() / scale
    if cache == "int8":
        return y.round().clamp(-128, 127).to(torch.int8)
    y = (y.round().clamp(-8, 7) + 8).to(torch.uint8)
    return y[..., 0::2] | (y[..., 1::2] << 4)


def _decode(codes, scale, cache):
    if cache == "fp8":
        return codes.double() * scale.double()
    if cache == "int8":
        return codes.double() * scale.double()
    lo, hi = (codes & 15).double() - 8, (codes >> 4).double() - 8
    return torch.stack((lo, hi), -1).flatten(-2) * scale.double()


def _inputs(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(int(seed))
    T = DTYPES[case["dtype"]]
    cache, kv, d = case["cache"], case["kv"], case["head"]
    lens = _lengths(case)
    B = len(lens)
    s = {"lens": lens, "k_scale": None, "v_scale": None}

    def normal(*shape, dtype=T):
        return torch.randn(shape, generator=g, device=dev, dtype=dtype)

    def uniform(*shape):
        return torch.rand(shape, generator=g, device=dev)

    def integer_scale():  # per channel, N(0, 1) rows filling the codes
        return (uniform(kv, d) * 0.5 + 0.75) * (4.0 / {"int8": 127, "int4": 7}[cache])

    if case["call"] == "gqa":
        S, cap = case["seq"], case["capacity"]
        s["total"] = max(n + p for n, p in lens)
        s["seqlens"] = np.array([n + p - 1 for n, p in lens], np.int32)
        s["query"] = normal(B, S, case["heads"] * d)
        s["key"], s["value"] = normal(B, S, kv * d), normal(B, S, kv * d)
        for side in ("key", "value"):
            if cap == 0:  # the presents that the call fills
                s[side + "_cache"] = torch.empty((B, kv, S, d), dtype=T, device=dev)
            elif cache == "same":
                s[side + "_cache"] = normal(B, kv, cap, d)
            else:
                s[side[0] + "_scale"] = sc = integer_scale()
                s[side + "_cache"] = torch.cat(
                    [_quantise(normal(kv, cap, d), sc[:, None], cache, True)[None]
                     for _ in range(B)])
        positions = max(cap, S)
    else:
        bs = case["block"]
        need = [-(-(n + p) // bs) for n, p in lens]
        nb, mb = sum(need) + 8, max(need)
        perm = np.random.default_rng(int(seed)).permutation(nb).astype(np.int32)
        bt = np.full((B, mb), perm[-1], np.int32)
        at = 0
        for b, n in enumerate(need):
            bt[b, :n] = perm[at:at + n]
            at += n
        s["block_table"] = bt
        s["cum"] = np.concatenate(([0], np.cumsum([n for n, _ in lens]))).astype(np.int32)
        s["past"] = np.array([p for _, p in lens], np.int32)
        tokens = int(s["cum"][-1])
        if case["call"] == "paged":
            s["query"] = normal(tokens, case["heads"] * d)
        s["key"] = normal(tokens, kv * d)
        s["value"] = None if case.get("latent") else normal(tokens, kv * d)
        for side in ("key", "value"):
            if s[side] is None:
                s[side + "_cache"] = None
            elif cache == "same":
                s[side + "_cache"] = normal(nb, bs, kv, d)
            elif cache == "fp8":  # one scale per (page, kv-head) from its largest value
                pages, scales = [], []
                for i in range(0, nb, 8192):
                    x = normal(min(8192, nb - i), bs, kv, d, dtype=torch.float32)
                    scales.append((x.abs().amax(dim=(1, 3)) / 448.0).clamp_min(1e-12))
                    pages.append(_quantise(x, scales[-1][:, None, :, None], cache))
                s[side + "_cache"], s[side[0] + "_scale"] = torch.cat(pages), torch.cat(scales)
            else:
                s[side[0] + "_scale"] = sc = integer_scale()
                s[side + "_cache"] = torch.cat(
                    [_quantise(normal(min(4096, nb - i), bs, kv, d), sc, cache)
                     for i in range(0, nb, 4096)])
        positions = max(n + p for n, p in lens)
    if case["call"] != "append":
        s["cos"] = s["sin"] = s["sink"] = s["q_norm"] = s["k_norm"] = None
        if case["rotary"]:
            half = case["rotary"] // 2
            inv = case["theta"] ** (-torch.arange(half, dtype=torch.float64, device=dev) / half)
            ang = torch.arange(positions, dtype=torch.float64, device=dev)[:, None] * inv
            s["cos"], s["sin"] = ang.cos().to(T), ang.sin().to(T)
        if case["sink"]:
            s["sink"] = normal(case["heads"])
        if case.get("norm"):
            s["q_norm"] = (1 + 0.1 * normal(d, dtype=torch.float32)).to(T)
            s["k_norm"] = (1 + 0.1 * normal(d, dtype=torch.float32)).to(T)
    return s


def _scale_attr(case):
    return 1.0 / math.sqrt(192.0) if case.get("latent") else 0.0  # 0: 1 / sqrt(head)


def prepare(case, seed):
    from onnxruntime_ep_mlx_amd import _capi as capi
    from onnxruntime_ep_mlx_amd import load, pa_dtype
    lib = load()
    s = _inputs(case, seed)
    dev = s["key"].device
    T = pa_dtype(DTYPES[case["dtype"]])
    quant = (capi.PA_QUANT_PER_CHANNEL if case["cache"] in ("int8", "int4")
             else capi.PA_QUANT_NONE)

    def ptr(t):
        return None if t is None else t.ctypes.data if isinstance(t, np.ndarray) else t.data_ptr()

    def device(a):
        s.setdefault("keep", []).append(torch.from_numpy(a).to(dev))
        return s["keep"][-1].data_ptr()

    B = len(s["lens"])
    if case["call"] == "gqa":
        s["out"] = torch.empty_like(s["query"])
        prompt = case["capacity"] == 0
        cos = s["cos"]
        node = capi.PaGqaNode(case["heads"], case["kv"], 0.0, case["softcap"], case["window"],
                              int(cos is not None), 0, 1, 1e-6, 0, 0, 0)
        io = capi.PaGqaIO(
            dtype=T, batch=B, seq=case["seq"], query_hidden=s["query"].shape[2],
            kv_seq=case["seq"], query=ptr(s["query"]), key=ptr(s["key"]), value=ptr(s["value"]),
            past_key=None if prompt else ptr(s["key_cache"]),
            past_value=None if prompt else ptr(s["value_cache"]), past_capacity=case["capacity"],
            present_key=ptr(s["key_cache"]), present_value=ptr(s["value_cache"]),
            present_capacity=s["key_cache"].shape[2], seqlens_k=device(s["seqlens"]),
            host_seqlens_k=ptr(s["seqlens"]), total_sequence_length=s["total"],
            cos_cache=ptr(cos), sin_cache=ptr(s["sin"]),
            rotary_positions=0 if cos is None else cos.shape[0],
            rotary_half=0 if cos is None else cos.shape[1], head_sink=ptr(s["sink"]),
            output=ptr(s["out"]),
            cache_dtype=0 if case["cache"] == "same" else pa_dtype(s["key_cache"].dtype),
            k_scale=ptr(s["k_scale"]), v_scale=ptr(s["v_scale"]), k_quant_type=quant,
            v_quant_type=quant)
        size, call = (lib.pa_group_query_attention_workspace_bytes, lib.pa_group_query_attention)
    else:
        nb, bs, kv, _ = s["key_cache"].shape
        cache = capi.PaCache(ptr(s["key_cache"]), ptr(s["value_cache"]), ptr(s["k_scale"]),
                             ptr(s["v_scale"]), nb, bs, kv, case["head"],
                             pa_dtype(s["key_cache"].dtype), quant, quant)
        tokens, mb = s["key"].shape[0], s["block_table"].shape[1]
        if case["call"] == "append":
            batch = capi.PaBatch(device(s["cum"]), device(s["past"]), device(s["block_table"]),
                                 None, B, mb, tokens, 0,
                                 capi.PA_BATCH_SLOTS_DISTINCT if case["distinct"] else 0, 0)
            args = (C.byref(cache), C.byref(batch), T, ptr(s["key"]), ptr(s["value"]))
            s["launch"] = lambda stream: capi.check(lib.pa_reshape_and_cache(*args, stream))
            return s
        s["out"] = torch.empty((tokens, case["heads"] * _v_head(case)), dtype=s["query"].dtype,
                               device=dev)
        cos = s["cos"]
        node = capi.PaNode(case["heads"], kv, _scale_attr(case), case["softcap"], case["window"],
                           int(cos is not None), 0, 512 if case["latent"] else 0, 1, 1e-6,
                           512 if case["latent"] else 0, int(case["latent"]))
        io = capi.PaIO(
            T, tokens, s["query"].shape[1], ptr(s["query"]), ptr(s["key"]), ptr(s["value"]), cache,
            device(s["cum"]), device(s["past"]), device(s["block_table"]), B, mb, ptr(cos),
            ptr(s["sin"]), 0 if cos is None else cos.shape[0], 0 if cos is None else cos.shape[1],
            None, ptr(s["sink"]), ptr(s["q_norm"]), ptr(s["k_norm"]), ptr(s["cum"]),
            ptr(s["past"]), ptr(s["block_table"]), None, ptr(s["out"]), None, None, 0, 0)
        size, call = lib.pa_paged_attention_workspace_bytes, lib.pa_paged_attention
    nbytes = size(C.byref(node), C.byref(io))
    s["workspace"] = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev)
    args = (C.byref(node), C.byref(io), s["workspace"].data_ptr(), nbytes)
    s["launch"] = lambda stream: capi.check(call(*args, stream))
    return s


def _as_output(cache):
    """A cache as an output: codes as bytes."""
    return cache.view(torch.uint8) if cache.element_size() == 1 else cache


def run(state):
    state["launch"](torch.cuda.current_stream().cuda_stream)
    outs = [] if "out" not in state else [state["out"]]
    return outs + [_as_output(state[n]) for n in ("key_cache", "value_cache")
                   if state[n] is not None]


# ---------------------------------------------------------------------------------- 64-bit result

def _norm(x, weight):
    y = x.double()
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6)
    return (y * weight.double()).to(x.dtype)


def _rope(x, cos, sin, offset):
    """Rotate-half on dims [offset, offset + 2 half); each operation rounds to the type of x."""
    half = cos.shape[-1]
    a, b = x[..., offset:offset + half], x[..., offset + half:offset + 2 * half]
    x = x.clone()
    cos, sin = cos[:, None], sin[:, None]
    x[..., offset:offset + half], x[..., offset + half:offset + 2 * half] = (
        a * cos - b * sin, b * cos + a * sin)
    return x


def _attend(case, q, k, v, past, sink):
    """q [n, H, d], k [L, kv, d], v [L, kv, vd] in 64 bits; row i at position past + i."""
    n, H, d = q.shape
    L, kv, vd = v.shape
    g = H // kv
    scale = _scale_attr(case) or 1.0 / math.sqrt(d)
    q = q.view(n, kv, g, d).transpose(0, 1).reshape(kv, n * g, d)
    sc = torch.matmul(q, k.permute(1, 2, 0).contiguous()) * scale
    if case["softcap"]:
        sc = case["softcap"] * torch.tanh(sc / case["softcap"])
    pos = past + torch.arange(n, device=q.device)
    key = torch.arange(L, device=q.device)
    seen = key[None] <= pos[:, None]
    if case["window"] > 0:
        seen &= key[None] > (pos.clamp_max(L - 1) - case["window"])[:, None]
    sc = sc.view(kv, n, g, L).masked_fill_(~seen[None, :, None], -math.inf)
    if sink is not None:
        extra = sink.double().view(kv, 1, g, 1).expand(kv, n, g, 1)
        p = torch.softmax(torch.cat((sc, extra), -1), -1)[..., :L]
    else:
        p = torch.softmax(sc, -1)
    o = torch.matmul(p.reshape(kv, n * g, L), v.transpose(0, 1).contiguous())
    return o.view(kv, n, g, vd).transpose(0, 1).reshape(n, H * vd)


def exact(case, seed):
    if case["call"] == "append":
        return None  # bytes: compared as they are
    s = _inputs(case, seed)
    H, kv, d, cache = case["heads"], case["kv"], case["head"], case["cache"]
    offset = 512 if case.get("latent") else 0
    gqa = case["call"] == "gqa"
    sides = ("key",) if s["value"] is None else ("key", "value")
    outs = []
    for b, (new, past) in enumerate(s["lens"]):
        total = past + new
        if gqa:
            q, rows = s["query"][b], {n: s[n][b][:new] for n in sides}
        else:
            i = int(s["cum"][b])
            q, rows = s["query"][i:i + new], {n: s[n][i:i + new] for n in sides}
        q = q.reshape(-1, H, d)
        rows = {n: r.reshape(new, kv, d) for n, r in rows.items()}
        if s["q_norm"] is not None:
            q, rows["key"] = _norm(q, s["q_norm"]), _norm(rows["key"], s["k_norm"])
        if s["cos"] is not None:
            at = past + torch.arange(q.shape[0], device=q.device)
            q = _rope(q, s["cos"][at], s["sin"][at], offset)
            rows["key"] = _rope(rows["key"], s["cos"][at[:new]], s["sin"][at[:new]], offset)
        whole = {}
        for n in sides:
            store, scale = s[n + "_cache"], s[n[0] + "_scale"]
            if gqa:
                if cache == "same":
                    store[b, :, past:total] = rows[n].transpose(0, 1)
                    if case["capacity"] == 0:
                        store[b, :, total:] = 0
                    whole[n] = store[b, :, :total].double().transpose(0, 1)
                else:
                    codes = _quantise(rows[n], scale, cache, True)
                    store[b, :, past:total] = codes.transpose(0, 1)
                    whole[n] = _decode(store[b, :, :total].transpose(0, 1), scale, cache)
                continue
            bs = case["block"]
            pos = torch.arange(total, device=q.device)
            table = torch.from_numpy(s["block_table"][b]).to(q.device).long()
            page, slot = table[pos // bs], pos % bs
            if cache == "fp8":
                sc = scale[page][..., None]
                raw = store.view(torch.uint8)
                raw[page[past:], slot[past:]] = _quantise(rows[n], sc[past:], cache).view(
                    torch.uint8)
                whole[n] = _decode(raw[page, slot].view(torch.float8_e4m3fn), sc, cache)
            elif cache == "same":
                store[page[past:], slot[past:]] = rows[n]
                whole[n] = store[page, slot].double()
            else:
                store[page[past:], slot[past:]] = _quantise(rows[n], scale, cache)
                whole[n] = _decode(store[page, slot], scale, cache)
        v = whole["value"] if "value" in whole else whole["key"][..., :_v_head(case)]
        outs.append(_attend(case, q.double(), whole["key"], v, past, s["sink"]))
    out = torch.stack(outs) if gqa else torch.cat(outs)
    return [out] + [s[n + "_cache"] if cache == "same" else None for n in sides]
