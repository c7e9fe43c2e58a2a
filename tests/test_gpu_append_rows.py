"""The chunked append (RMSNorm + RoPE + cache store, 16 bytes per lane) against the per-row kernel:
the same call with and without the distinct-slots promise must leave the same bytes everywhere."""
import ctypes as C

import numpy as np
import pytest

import _oracle as orc
from pa_cases import from_torch, rotary_cache, to_torch

pytestmark = pytest.mark.gpu

# heads, kv, head, rotary dims, offset, interleaved, norm
FORMS = [
    (8, 2, 64, 64, 0, 0, False), (5, 1, 64, 32, 16, 1, True), (7, 7, 128, 128, 0, 0, True),
    (4, 2, 128, 48, 8, 0, False), (6, 2, 256, 64, 0, 0, True), (3, 1, 256, 256, 0, 1, False),
    (6, 3, 96, 96, 0, 0, False), (5, 1, 576, 64, 512, 0, False), (3, 1, 200, 16, 184, 1, False),
    (4, 2, 128, 20, 0, 1, False), (4, 2, 128, 0, 0, 0, True), (4, 2, 80, 0, 0, 0, False),
]


def _append(form, new_lens, dtype, cache, distinct, in_place=False, skip=False, seed=1):
    import torch
    from onnxruntime_ep_mlx_amd import _capi as capi
    heads, kv, d, rot, off, inter, norm = form
    rng = np.random.default_rng(seed)
    B, bs, cap = len(new_lens), 16, 512
    past = rng.integers(0, cap - max(new_lens), size=B).astype(np.int32)
    cum = np.concatenate([[0], np.cumsum(new_lens)]).astype(np.int32)
    T, mb = int(cum[-1]), cap // bs
    bt = rng.permutation(B * mb).astype(np.int32).reshape(B, mb)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    draw = lambda *s: to_torch(orc.encode(rng.standard_normal(s), dtype), dtype)
    q, k, v = draw(T, heads * d), draw(T, kv * d), draw(T, kv * d)
    width = (d + 1) // 2 if cache == orc.I4 else d
    shape = (B * mb, bs, kv, width)
    if cache == dtype:
        kc, vc = draw(*shape), draw(*shape)
    else:
        tt = {orc.E4M3: torch.float8_e4m3fn, orc.I8: torch.int8, orc.I4: torch.uint8}[cache]
        kc, vc = (dev(rng.integers(0, 100, shape).astype(np.uint8)).view(tt) for _ in range(2))
    scale = lambda: dev(np.abs(rng.standard_normal(
        (B * mb, kv) if cache == orc.E4M3 else (kv, d))).astype(np.float32) / 40)
    ks, vs = (scale(), scale()) if cache != dtype else (None, None)
    if ks is not None:
        ks.view(-1)[3] = 0.0  # a zero scale stores zero codes
    cos = sin = None
    if rot:
        cos, sin = (to_torch(t, dtype) for t in rotary_cache(cap + 8, rot, 10000.0, dtype))
    qn = kn = None
    if norm:
        qn, kn = draw(d), draw(d)
    slots = None
    if skip:  # explicit slots, some of them skipped
        pos = np.concatenate([past[b] + np.arange(n) for b, n in enumerate(new_lens)])
        seq = np.repeat(np.arange(B), new_lens)
        s = bt[seq, pos // bs] * bs + pos % bs
        s[::3] = -1
        slots = dev(s.astype(np.int32))
    transform = bool(rot or norm)
    qo = (q if in_place else torch.zeros_like(q)) if transform else None
    ko = (k if in_place else torch.zeros_like(k)) if transform else None
    ptr = lambda t: None if t is None else t.data_ptr()
    tcum, tpast, tbt = dev(cum), dev(past), dev(bt)
    codes = {orc.E4M3: capi.PA_DTYPE_FP8_E4M3, orc.I8: capi.PA_DTYPE_INT8,
             orc.I4: capi.PA_DTYPE_INT4}
    act = capi.PA_DTYPE_BFLOAT16 if dtype == orc.BF16 else capi.PA_DTYPE_FLOAT16
    quant = 2 if cache in (orc.I8, orc.I4) else 0
    cd = capi.PaCache(ptr(kc), ptr(vc), ptr(ks), ptr(vs), B * mb, bs, kv, d,
                      codes.get(cache, act), quant, quant)
    bd = capi.PaBatch(ptr(tcum), ptr(tpast), ptr(tbt), ptr(slots), B, mb, T, 0,
                      capi.PA_BATCH_SLOTS_DISTINCT if distinct else 0, 0)
    capi.check(capi.load().pa_rotary_append(
        C.byref(cd), C.byref(bd), heads, act, ptr(q), ptr(k), ptr(v), ptr(qo), ptr(ko), ptr(cos),
        ptr(sin), cos.shape[0] if rot else 0, rot // 2, off, inter, ptr(qn), ptr(kn), 1e-6,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return [t.view(torch.uint8).cpu().numpy() for t in (qo, ko, kc, vc) if t is not None]


def _same(a, b):
    assert all(np.array_equal(x, y) for x, y in zip(a, b)) and len(a) == len(b)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype", [orc.BF16, orc.F16])
@pytest.mark.parametrize("new_lens", [[1], [1, 3, 1, 2, 1], [17, 1, 400, 63]])
def test_same_bytes_as_the_per_row_kernel(form, dtype, new_lens):
    _same(*(_append(form, new_lens, dtype, dtype, d) for d in (True, False)))


@pytest.mark.parametrize("cache", [orc.E4M3, orc.I8, orc.I4])
@pytest.mark.parametrize("form", [f for f in FORMS if f[2] in (64, 128, 256, 200)])
def test_same_codes_as_the_per_row_kernel(form, cache):
    _same(*(_append(form, [5, 1, 90], orc.BF16, cache, d) for d in (True, False)))


@pytest.mark.parametrize("form", [FORMS[2], FORMS[4], FORMS[6], FORMS[7]])
def test_in_place_and_skipped_slots(form):
    want = _append(form, [31, 1, 70], orc.BF16, orc.BF16, False, skip=True)
    _same(_append(form, [31, 1, 70], orc.BF16, orc.BF16, True, skip=True), want)
    _same(_append(form, [31, 1, 70], orc.BF16, orc.BF16, True, in_place=True, skip=True), want)


@pytest.mark.parametrize("dtype", [orc.BF16, orc.F16])
@pytest.mark.parametrize("heads,d", [(8, 64), (4, 128), (3, 256), (3, 96)])
def test_norm_rows_against_the_oracle(dtype, heads, d):
    """Normalised query rows bit for bit (each product rounded on its own): 1600 rows and more, as
    a fused rounding differs about once in 25,000 elements."""
    import torch
    import onnxruntime_ep_mlx_amd as ep
    rng = np.random.default_rng(d)
    T = 600
    enc = lambda *s: orc.encode(rng.standard_normal(s), dtype)
    q, k, wq, wk = enc(T, heads * d), enc(T, d), enc(d), enc(d)
    dev = lambda a: to_torch(a, dtype)
    kc = torch.zeros((T // 16 + 1, 16, 1, d), dtype=dev(q).dtype, device="cuda")
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    for distinct in (True, False):
        got, _ = ep.rotary_append(
            dev(q), dev(k), dev(k), kc, kc.clone(), i32([0, T]), i32([0]),
            i32([list(range(T // 16 + 1))]), num_heads=heads, q_norm_weight=dev(wq),
            k_norm_weight=dev(wk), slots_distinct=distinct)
        want = orc.rms_norm_rows(q, heads, d, wq, 1e-6, dtype)
        assert np.array_equal(from_torch(got, dtype).reshape(-1), want.reshape(-1))
