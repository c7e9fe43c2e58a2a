"""Workspace sizing of multi-token batches over operand images (host only, no GPU).

The planned prefill writes operand images (fp16 key and value rows laid out as the kernel's LDS
operands, 32 KiB per 64-key step of every (sequence, kv-head) at head 128) into the workspace.
They are sized by the live context of the call -- the host metadata's longest past + new tokens,
the caller's max_context_len, or GroupQueryAttention's total_sequence_length -- not by the
block-table or present capacity.  These cases check that the image region is planned and has the
live size, and that a region beyond the 2 GiB image limit (byte-coded pages: int8 / int4 / fp8)
is planned for groups of sequences that fit it rather than dropped.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from onnxruntime_ep_mlx_amd import _capi as capi

FAKE = 0x1000  # device pointers are never dereferenced by the size queries
STEP_BYTES = 2 * 64 * 128 * 2  # one 64-key image step at head 128 (keys + values, fp16)


def _gqa(total, cap, B=8, S=512, H=32, KV=8, d=128, cache=capi.PA_DTYPE_INT8):
    host = np.full(B, total - 1, np.int32)
    node = capi.PaGqaNode(H, KV, 0.0, 0.0, -1, 0, 0, 1, 1e-6, 0)
    io = capi.PaGqaIO(dtype=capi.PA_DTYPE_BFLOAT16, batch=B, seq=S, query_hidden=H * d,
                      kv_seq=S, query=FAKE, key=FAKE, value=FAKE, past_key=FAKE,
                      past_value=FAKE + 64, past_capacity=cap, present_key=FAKE,
                      present_value=FAKE + 64, present_capacity=cap, seqlens_k=FAKE,
                      host_seqlens_k=host.ctypes.data, total_sequence_length=total,
                      output=FAKE, cache_dtype=cache, k_scale=FAKE, v_scale=FAKE,
                      k_quant_type=capi.PA_QUANT_PER_CHANNEL,
                      v_quant_type=capi.PA_QUANT_PER_CHANNEL)
    return node, io, host


def test_gqa_integer_present_images_follow_total_not_capacity():
    """Advisor case: batch 8, kv 8, capacity 131072, head 128, a 2048-key call: the images are
    8 * 8 * 32 steps (64 MiB), not 8 * 8 * 2048 steps (4 GiB, beyond the image limit)."""
    lib = capi.load()
    B, KV, total, cap = 8, 8, 2048, 131072
    node, io, keep = _gqa(total, cap, B=B, KV=KV)
    n = lib.pa_group_query_attention_workspace_bytes(C.byref(node), C.byref(io))
    live = B * KV * (total // 64) * STEP_BYTES
    assert live <= n < live + (256 << 20), n
    # the same call at a small capacity plans the same images
    node2, io2, keep2 = _gqa(total, total, B=B, KV=KV)
    n2 = lib.pa_group_query_attention_workspace_bytes(C.byref(node2), C.byref(io2))
    assert abs(n - n2) < (1 << 20), (n, n2)


def _paged(past, nq, max_blocks, bs=16, KV=8, H=64, d=128, host=True, bound=0,
           cache=capi.PA_DTYPE_FP8_E4M3, act=capi.PA_DTYPE_BFLOAT16, window=-1):
    B = len(past)
    cum = np.concatenate([[0], np.cumsum([nq] * B)]).astype(np.int32)
    past = np.asarray(past, np.int32)
    nb = B * max_blocks
    bt = np.arange(nb, dtype=np.int32).reshape(B, max_blocks)
    keep = [cum, past, bt]
    c = capi.PaCache(FAKE, FAKE, FAKE, FAKE, nb, bs, KV, d, cache)
    T = int(cum[-1])
    io = capi.PaIO(act, T, H * d, FAKE, FAKE, FAKE, c, FAKE, FAKE, FAKE,
                   B, max_blocks, None, None, 0, 0, None, None, None, None,
                   cum.ctypes.data if host else None, past.ctypes.data if host else None,
                   bt.ctypes.data if host else None, None, FAKE, None, None,
                   nq if not host else 0, bound)
    node = capi.PaNode(H, KV, 0.0, 0.0, window, 0, 0, 0, 1, 1e-6)
    return node, io, keep


def test_paged_fp8_images_follow_live_context_with_host_metadata():
    """fp8 pages, batch 16, kv 8, a 65,536-position block table (4096 pages of 16) and live
    contexts of at most 1,064 keys: 17 image steps per (sequence, kv-head)."""
    lib = capi.load()
    past = [1000, 40, 700, 3] * 4
    node, io, keep = _paged(past, 64, 4096)
    n = lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io))
    live = 16 * 8 * -(-(1000 + 64) // 64) * STEP_BYTES
    assert live <= n < live + (256 << 20), n


def test_paged_images_follow_the_callers_context_bound():
    lib = capi.load()
    past = [1000, 40, 700, 3] * 4
    node, io, keep = _paged(past, 64, 4096, host=False, bound=1064)
    n = lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io))
    live = 16 * 8 * 17 * STEP_BYTES
    assert live <= n < live + (256 << 20), n
    # without a bound the images cover the block-table capacity (65,536 positions: 1,024 steps,
    # 256 MiB per sequence), 4 GiB for the batch: the planned launch runs on groups of 8
    # sequences, the workspace holding the images of one group (2 GiB) and its plan
    node0, io0, keep0 = _paged(past, 64, 4096, host=False, bound=0)
    n0 = lib.pa_paged_attention_workspace_bytes(C.byref(node0), C.byref(io0))
    group = 8 * 8 * 1024 * STEP_BYTES
    assert group == 1 << 31
    assert group <= n0 < group + (64 << 20), n0


def test_context_bound_below_the_host_metadata_is_refused():
    lib = capi.load()
    node, io, keep = _paged([1000, 40], 64, 128, bound=500)
    rc = lib.pa_paged_attention(C.byref(node), C.byref(io), C.c_void_p(0x2000), 1 << 40, None)
    msg = lib.pa_last_error().decode()
    assert rc == capi.PA_ERR_INVALID_ARGUMENT and "max_context_len" in msg, msg
    node, io, keep = _paged([1000, 40], 64, 128, bound=-1)
    rc = lib.pa_paged_attention(C.byref(node), C.byref(io), C.c_void_p(0x2000), 1 << 40, None)
    assert rc == capi.PA_ERR_INVALID_ARGUMENT


def test_short_prefills_plan_images_of_a_bounded_context_only():
    """5 prompts of 100 tokens (160 row blocks, below the workgroup slots) over a 32,768-position table:
    without a bound on their contexts the call keeps the grid launch and asks for no images (5 x 8 x 512
    steps); with host metadata or a bound it may plan them."""
    lib = capi.load()

    def size(**kw):
        node, io, keep = _paged([1900] * 5, 100, 2048, H=32, cache=capi.PA_DTYPE_BFLOAT16, **kw)
        return lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io))

    images = 5 * 8 * 32 * STEP_BYTES
    partials = 500 * 32 * 128 * 4 * 5  # fp32 rows of at most 5 chunks
    assert size(host=False) < partials
    assert images <= size(host=True) < images + (100 << 20)
    assert size(host=False, bound=2000) == size(host=True)


# heads, kv-heads, head, sequences, new tokens, past, window, table positions (0: what is needed); both
# launches timed on an MI355X, us, planned / grid
@pytest.mark.parametrize("H,KV,d,B,nq,past,window,table,planned", [
    (32, 8, 128, 60, 29, 1000, -1, 0, False),   # 197 / 141: images read by one row block each
    (32, 8, 128, 38, 29, 3000, 128, 0, False),  # 233 / 64: of keys that no row sees
    (32, 8, 128, 15, 125, 3000, 128, 0, False),  # 129 / 87
    (64, 8, 64, 38, 13, 3000, 128, 0, False),   # 125 / 53
    (32, 8, 128, 4, 125, 3000, -1, 0, False),   # 87 / 75
    (32, 8, 128, 2, 512, 1000, -1, 0, True),    # 73 / 84
    (32, 8, 128, 1, 2000, 4000, 128, 0, True),  # 52 / 86: a window over many row blocks
    (64, 8, 64, 8, 45, 1000, -1, 0, True),      # 45 / 65
    (32, 8, 128, 6, 125, 1000, 128, 0, True),   # 42 / 62: few keys an item, no parts
    (32, 8, 128, 4, 125, 1000, -1, 8960, True),  # 55 / 69: chunks cut from a table of 8 contexts
])
def test_short_prefills_weigh_images_against_what_reads_them(H, KV, d, B, nq, past, window, table,
                                                             planned):
    lib = capi.load()
    for act in (capi.PA_DTYPE_BFLOAT16, capi.PA_DTYPE_FLOAT16):
        n = []
        for host in (True, False):  # without a bound: the grid launch
            node, io, keep = _paged([past] * B, nq, max(-(-(past + nq) // 16), table // 16), KV=KV,
                                    H=H, d=d, host=host, cache=act, act=act, window=window)
            n.append(lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io)))
        assert (n[0] != n[1]) == planned


@pytest.mark.parametrize("past,planned", [(0, False), (3000, True)])  # 48 / 60 us planned / grid
def test_short_prefills_weigh_the_batch_by_its_sequences(past, planned):
    """7 prompts of 45 tokens without a past and one with: the grid launch cuts every sequence into
    chunks of the longest context's table, the images hold what is there."""
    lib = capi.load()
    n = []
    for host in (True, False):
        node, io, keep = _paged([0] * 7 + [past], 45, -(-(past + 45) // 16), H=32, host=host,
                                cache=capi.PA_DTYPE_BFLOAT16)
        n.append(lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io)))
    assert (n[0] != n[1]) == planned


def test_forced_prefill_kind_splits_short_batches_over_the_grid():
    """pa_attention_ex with kind 2: the planned launch once the batch fills the GPU, else context chunks;
    the automatic choice may plan a short batch over images."""
    lib = capi.load()
    B, nq, past, KV, H, d, bs = 2, 512, 1000, 8, 32, 128, 16
    mb = -(-(past + nq) // bs)
    cache = capi.PaCache(FAKE, FAKE, None, None, B * mb, bs, KV, d, capi.PA_DTYPE_BFLOAT16)
    batch = capi.PaBatch(FAKE, FAKE, FAKE, None, B, mb, B * nq, nq, 0, past + nq)
    attn = capi.PaAttn(H, 0.0, 0.0, -1, 1, None)
    size = lambda kind: lib.pa_attention_workspace_bytes_ex(
        C.byref(cache), C.byref(batch), C.byref(attn), capi.PA_DTYPE_BFLOAT16, kind, 0)
    chunks = 2  # 256 row blocks, 512 workgroup slots
    partials = B * nq * H * chunks * (d * 4 + 8)
    assert partials <= size(2) < partials + 1024
    assert size(0) > B * KV * 24 * STEP_BYTES


def _latent(past, H, table=0, bs=16, nq=1, host=True):
    B = len(past)
    cum = (np.arange(B + 1) * nq).astype(np.int32)
    past = np.asarray(past, np.int32)
    mb = -(-max(int(past.max()) + nq, table) // bs)
    cache = capi.PaCache(FAKE, None, None, None, B * mb, bs, 1, 576, capi.PA_DTYPE_BFLOAT16)
    io = capi.PaIO(capi.PA_DTYPE_BFLOAT16, B * nq, H * 576, FAKE, FAKE, None, cache, FAKE, FAKE, FAKE, B,
                   mb, None, None, 0, 0, None, None, None, None, cum.ctypes.data if host else None,
                   past.ctypes.data if host else None, FAKE if host else None, None, FAKE, None, None,
                   0 if host else nq, 0)
    node = capi.PaNode(H, 1, 192.0**-0.5, 0.0, -1, 0, 0, 0, 1, 1e-6, 512, 1)
    return capi.load().pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io))


SEGMENTS = 2 * 256 * 64 * (512 * 4 + 8) + 256 * 16  # partials and list of the 64-row blocks


# heads, sequences, keys; 64-row blocks / smaller ones, us on an MI355X
@pytest.mark.parametrize("H,B,keys,wide", [
    (16, 4, 64, False),    # 18.3 / 16.2
    (16, 64, 96, False),   # 23.4 / 19.0
    (16, 64, 128, False),  # 23.5 / 20.9
    (16, 4, 128, True),    # 18.9 / 19.5
    (16, 64, 256, True),   # 27.3 / 28.6
    (32, 64, 96, True),    # 29.7 / 30.0
    (128, 16, 96, False),  # 33.5 / 29.7
    (64, 32, 128, False),  # 33.2 / 31.8
    (128, 8, 96, True),    # 26.9 / 27.8
    (128, 48, 192, False),  # 51.3 / 40.8
    (128, 32, 192, True),  # 37.5 / 38.5
    (128, 64, 384, False),  # 59.7 / 55.4
    (128, 64, 448, True),
    (128, 66, 256, True),  # more than one round of the smaller blocks
])
def test_latent_blocks_follow_rows_and_keys(H, B, keys, wide):
    n = _latent([keys - 1] * B, H)
    assert (n == SEGMENTS) == wide, n


def test_latent_blocks_of_short_contexts_behind_a_long_table():
    """The smaller blocks' grid covers the table: 16 heads, 4 contexts of 64 keys behind 8192."""
    assert _latent([63] * 4, 16, table=8192) == SEGMENTS


def test_latent_segments_are_asked_for_only_where_they_can_run():
    """The 64-row blocks read every row from the pages: without host metadata (operator) or
    PA_BATCH_NEW_ROWS_IN_CACHE (kernel entry), or with a slot mapping, they cannot run."""
    lib = capi.load()
    assert _latent([1000] * 4, 16) == SEGMENTS
    assert _latent([1000] * 4, 16, host=False) < SEGMENTS // 8
    cache = capi.PaCache(FAKE, None, None, None, 256, 16, 1, 576, capi.PA_DTYPE_BFLOAT16)
    attn = capi.PaAttn(16, 0.1, 0.0, -1, 1, None, 512)
    for flags, slots, wide in ((0, None, False), (capi.PA_BATCH_NEW_ROWS_IN_CACHE, None, True),
                               (capi.PA_BATCH_NEW_ROWS_IN_CACHE, FAKE, False)):
        batch = capi.PaBatch(FAKE, FAKE, FAKE, slots, 4, 64, 4, 1, flags, 0)
        n = lib.pa_attention_workspace_bytes_ex(C.byref(cache), C.byref(batch), C.byref(attn),
                                                capi.PA_DTYPE_BFLOAT16, 0, 0)
        assert (n == SEGMENTS) == wide, (flags, n)


# decode sequences and their contexts beside one prompt after 2000 keys; split / whole, us
@pytest.mark.parametrize("kv,d,steps,past,nq,window,split", [
    (8, 128, 16, 3000, 30, -1, False),  # 71 / 53: a prompt of one row block
    (8, 128, 48, 3000, 30, -1, True),   # 123 / 141
    (8, 128, 16, 3000, 40, -1, True),   # two row blocks
    (4, 128, 16, 3000, 40, -1, False),  # 61 / 50: fewer key rows
    (4, 128, 16, 8000, 40, -1, True),
    (8, 128, 4, 8000, 96, -1, True),    # 54 / 73
    (8, 96, 16, 3000, 30, -1, False),
    (8, 96, 48, 3000, 30, -1, True),
    (8, 128, 16, 400, 130, -1, False),  # too few keys
    (8, 128, 48, 300, 30, -1, False),   # nor over images, most of whose workgroups find no keys: 86 / 64
    (8, 128, 16, 3000, 30, 1024, False),  # the whole contexts count
    (8, 128, 16, 8000, 30, 1024, True),   # 45 / 54
])
def test_mixed_batches_split_by_the_keys_and_the_prompts_blocks(kv, d, steps, past, nq, window, split):
    lib = capi.load()
    cum = np.concatenate([np.arange(steps + 1), [steps + nq]]).astype(np.int32)
    past = np.array([past] * steps + [2000], np.int32)
    mb = -(-int((past + np.diff(cum)).max()) // 16)
    dt = capi.PA_DTYPE_BFLOAT16
    heads = 4 * kv
    cache = capi.PaCache(FAKE, FAKE, None, None, (steps + 1) * mb, 16, kv, d, dt)
    io = capi.PaIO(dt, int(cum[-1]), heads * d, FAKE, FAKE, FAKE, cache, FAKE, FAKE, FAKE, steps + 1, mb, None,
                   None, 0, 0, None, None, None, None, cum.ctypes.data, past.ctypes.data, FAKE, None, FAKE,
                   None, None, 0, 0)
    node = capi.PaNode(heads, kv, 0.0, 0.0, window, 0, 0, 0, 1, 1e-6)
    n = [lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io))]
    io.host_cumulative_sequence_length = io.host_past_seqlens = None  # whole, on its plain plan
    io.max_query_len = nq
    n.append(lib.pa_paged_attention_workspace_bytes(C.byref(node), C.byref(io)))
    decode = kv * 16 * 128 * (d * 4 + 8)  # partials of the streaming decode's segments, at the least
    assert (n[0] >= decode and n[0] > n[1]) == split, n
