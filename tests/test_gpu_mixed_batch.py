"""Decode and prefill sequences in one batch: with host metadata the call runs each kind on its own
kernels.  Against a float64 evaluation of every sequence over the updated pages, and against the same
batch without host metadata (one prefill launch): the pages byte for byte."""
import ctypes as C

import numpy as np
import pytest

import onnxruntime_ep_mlx_amd as ep

pytestmark = pytest.mark.gpu


class Mixed:
    def __init__(self, heads, kv, head, block, new, past, dtype="bfloat16", cache=None, rot=0,
                 window=-1, softcap=0.0, sink=False):
        import torch
        g = torch.Generator(device="cuda").manual_seed(len(new) + head)
        T = getattr(torch, dtype)
        self.new, self.past, self.block, self.cache = new, past, block, cache
        need = [-(-(n + p) // block) for n, p in zip(new, past)]
        perm = np.random.default_rng(head).permutation(sum(need) + 3).astype(np.int32)
        bt, at = np.full((len(new), max(need)), perm[-1], np.int32), 0
        for i, n in enumerate(need):
            bt[i, :n] = perm[at:at + n]
            at += n
        self.bt = torch.from_numpy(bt).cuda()
        self.cum = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
        t = int(self.cum[-1])
        rnd = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=T)
        self.q, self.k, self.v = rnd(t, heads * head), rnd(t, kv * head), rnd(t, kv * head)
        shape = (len(perm), block, kv, head)
        self.scales = {}
        if cache is None:
            self.pages = [rnd(*shape), rnd(*shape)]
        elif cache == "fp8":
            self.pages = [rnd(*shape).clamp(-3, 3).to(torch.float8_e4m3fn) for _ in "kv"]
            self.scales = {n + "_scale": torch.rand((len(perm), kv), generator=g, device="cuda")
                           + 0.5 for n in "kv"}
        else:
            width = head if cache == "int8" else head // 2
            bits = torch.int8 if cache == "int8" else torch.uint8
            lo, hi = (-100, 100) if cache == "int8" else (0, 256)
            self.pages = [torch.randint(lo, hi, (*shape[:3], width), generator=g, device="cuda",
                                        dtype=bits) for _ in "kv"]
            unit = 50.0 if cache == "int8" else 4.0
            self.scales = {n + "_scale": (torch.rand((kv, head), generator=g, device="cuda") + 0.5)
                           / unit for n in "kv"}
            self.scales.update(k_quant_type="PER_CHANNEL", v_quant_type="PER_CHANNEL")
        self.cos = self.sin = None
        if rot:
            inv = 1e4 ** (-torch.arange(rot // 2, device="cuda").double() * 2 / rot)
            ang = torch.arange(max(n + p for n, p in zip(new, past)), device="cuda")[:, None] * inv
            self.cos, self.sin = ang.cos().to(T), ang.sin().to(T)
        self.sink = rnd(heads) if sink else None
        self.opts = dict(num_heads=heads, kv_num_heads=kv, local_window_size=window,
                         softcap=softcap, do_rotary=int(rot > 0))

    def call(self, **kw):
        import torch
        k, v = (p.clone() for p in self.pages)
        i32 = lambda a: torch.tensor(np.asarray(a, np.int32)).cuda()
        out, k, v = ep.paged_attention(self.q, self.k, self.v, k, v, i32(self.cum), i32(self.past),
                                       self.bt, self.cos, self.sin, head_sink=self.sink,
                                       **self.scales, **self.opts, **kw)
        torch.cuda.synchronize()
        return out, k, v

    def rows(self, pages, side, b, n):
        """Keys or values [n, kv, head] of sequence b in float64."""
        import torch
        pos = torch.arange(n, device="cuda")
        page = self.bt[b].long()[pos // self.block]
        if self.cache is None:
            return pages[page, pos % self.block].double()
        sc = self.scales[side + "_scale"]
        raw = pages.view(torch.uint8)[page, pos % self.block]
        if self.cache == "fp8":
            return raw.view(torch.float8_e4m3fn).double() * sc[page][..., None]
        if self.cache == "int8":
            return raw.view(torch.int8).double() * sc
        return torch.stack(((raw & 15).double() - 8, (raw >> 4).double() - 8), -1).flatten(-2) * sc

    def check(self, out, k, v):
        import torch
        H, kv = self.opts["num_heads"], self.opts["kv_num_heads"]
        d, g = self.q.shape[1] // H, H // kv
        for b, (n, past) in enumerate(zip(self.new, self.past)):
            if n == 0:
                continue
            q = self.q[self.cum[b]:self.cum[b + 1]].view(n, H, d)
            if self.cos is not None:
                c, s = (t[past:past + n, None] for t in (self.cos, self.sin))
                h = c.shape[-1]
                x, y = q[..., :h], q[..., h:2 * h]
                q = torch.cat((x * c - y * s, y * c + x * s, q[..., 2 * h:]), -1)
            keys, vals = self.rows(k, "k", b, past + n), self.rows(v, "v", b, past + n)
            s = torch.einsum("nkgd,lkd->kgnl", q.double().view(n, kv, g, d), keys) * d ** -0.5
            if self.opts["softcap"]:
                s = self.opts["softcap"] * torch.tanh(s / self.opts["softcap"])
            row = past + torch.arange(n, device="cuda")[:, None]
            col = torch.arange(past + n, device="cuda")[None]
            seen = col <= row
            if self.opts["local_window_size"] > 0:
                seen &= col > row - self.opts["local_window_size"]
            s = s.masked_fill(~seen, -np.inf)
            if self.sink is not None:
                extra = self.sink.double().view(kv, g, 1, 1).expand(kv, g, n, 1)
                p = torch.softmax(torch.cat((s, extra), -1), -1)[..., :-1]
            else:
                p = torch.softmax(s, -1)
            want = torch.einsum("kgnl,lkd->nkgd", p, vals).reshape(n, H * d)
            got = out[self.cum[b]:self.cum[b + 1]].double()
            # one rounding to T: at most 2^-9 (bf16) or 2^-12 (fp16) of each element; fp16
            # probabilities (2^-12) and coded pages' fp16 queries and keys (2^-11) on top
            assert ((got - want).norm() / want.norm()).item() <= 4e-3, b


# heads, kv, head, block, new tokens, past: the decode sequences hold 240 MB and more of 16-bit keys
# and values (the last two 64 to 70), the others run the grid launch or (more rows) the planned one
SHAPES = [
    (32, 8, 128, 16, [1, 1, 40, 1, 0, 2, 1, 300], [13900, 16201, 33, 15640, 50, 777, 15500, 0]),
    (16, 2, 64, 16, [1] * 70 + [513, 1, 129], [6800] * 70 + [64, 1, 2000]),  # ranks past 64
    (8, 2, 256, 32, [1, 200, 1, 3, 4], [60000, 100, 30999, 31, 32040]),
    (8, 4, 96, 16, [700, 1, 1, 900, 1], [0, 82500, 81801, 300, 2000]),
    (28, 4, 128, 16, [2, 1, 513, 600, 512, 64, 1], [61000, 62999, 700, 0, 1300, 5, 1]),
    (64, 8, 64, 16, [1000, 900, 800, 1, 1], [0, 10, 500, 63100, 61000]),
    (32, 8, 128, 16, [1] * 20 + [400], [800] * 20 + [3]),
    (24, 4, 256, 256, [1, 130, 2, 1], [5000, 900, 5300, 5200]),
]
FORMS = [dict(rot=32), dict(dtype="float16", window=31000, softcap=20.0, sink=True)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_batch(shape, form):
    m = Mixed(*shape, **form)
    got, whole = m.call(), m.call(validate=False)
    assert all((a == b).all() for a, b in zip(got[1:], whole[1:]))
    m.check(*got)
    m.check(*whole)


@pytest.mark.parametrize("cache", ["fp8", "int8", "int4"])
@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[4]])
def test_mixed_batch_over_coded_pages(shape, cache):
    m = Mixed(*shape, cache=cache, rot=64)
    m.check(*m.call())


def test_workspace_sized_without_host_metadata_is_enough(monkeypatch):
    """A caller may size the workspace by its bounds alone: the batch then runs unsplit."""
    m = Mixed(*SHAPES[0])
    lib, seen = ep.load(), []
    size = lib.pa_paged_attention_workspace_bytes

    class Lib:
        def __getattr__(self, name):
            return getattr(lib, name)

        def pa_paged_attention_workspace_bytes(self, node, io):
            plain = type(io._obj).from_buffer_copy(io._obj)
            plain.host_cumulative_sequence_length = plain.host_past_seqlens = None
            plain.max_query_len = max(m.new)
            plain.max_context_len = max(n + p for n, p in zip(m.new, m.past))
            seen.append(size(node, C.byref(plain)))
            return seen[-1]

    monkeypatch.setattr(ep._capi, "load", Lib)
    m.check(*m.call())
    assert len(seen) == 1
