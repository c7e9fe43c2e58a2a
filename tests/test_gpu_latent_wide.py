"""LATENT caches of MLA rows (576 dims, values = the first 512) in blocks of 64 grouped query rows: the
edges of a block's two 32-row tiles, of a 64-key step and of a segment, against the oracle.

Bars: key cache bytes bit-exact.  Outputs: both sides are rounded to T, and the fp32 sums before that
differ by far less than a step of T, so few elements differ, by one step: the whole must stay below the
rounding itself, a step / sqrt(12) at values in [1, 2).
"""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as orc
from _oracle import BF16, F16
from pa_cases import make_latent_case, run_gpu_op

pytestmark = pytest.mark.gpu
TOL = {BF16: 2.0**-7 / 12**0.5, F16: 2.0**-10 / 12**0.5}


def check(H, new, past, bs=16, dtype=BF16, static=False, **kw):
    B = len(new)
    mb = -(-max(p + n for p, n in zip(past, new)) // bs) + 1
    c = make_latent_case(H, 576, 512, B * mb, bs, B, dtype=dtype, seed=H + B + sum(past) % 1000,
                         new_lens=list(new), past=np.array(past), max_blocks=mb, do_rotary=1,
                         rot_dim=64, rotary_offset=512, scale=kw.pop("scale", 192.0**-0.5), std=1.0,
                         **kw)
    print(f"latent wide H={H} new={new[:6]} past={past[:6]} bs={bs} dtype={dtype}", flush=True)
    ref, _, kc_ref, _ = orc.paged_attention_op(c)
    out, kc, _ = run_gpu_op(c, static_scratch=static)
    np.testing.assert_array_equal(kc, kc_ref)
    want = orc.decode(orc.encode(ref.astype(np.float32), dtype), dtype).astype(np.float64)
    err = orc.rel_l2(orc.decode(out, dtype).astype(np.float64), want)
    assert err <= TOL[dtype], err


@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("H,new", [(16, [1]), (32, [1, 1]), (33, [1]), (64, [1, 1, 1]), (65, [1]),
                                   (24, [3, 1]), (16, [5, 70]), (128, [1, 2])])
def test_row_blocks(H, new, dtype):
    check(H, new, [130 + 67 * i for i in range(len(new))], dtype=dtype)


@pytest.mark.parametrize("bs", [16, 32, 64])
def test_step_edges(bs):
    past = [0, 1, 14, 15, 16, 31, 46, 62, 63, 64, 95, 126, 127, 128, 190, 255]
    check(32, [1] * len(past), past, bs=bs)


# one pair over every segment (its partials merged by groups), few pairs, more pairs than segments
@pytest.mark.parametrize("H,past", [(16, [17000]), (128, [6390, 4000]),
                                    (16, [40 + 5 * i for i in range(300)]),
                                    (64, [(37 * i) % 900 for i in range(64)])],
                         ids=["one", "few", "more", "batch"])
def test_segments(H, past):
    check(H, [1] * len(past), past)


@pytest.mark.parametrize("window,softcap,sink,scale", [(100, 0.0, False, 0.07), (-1, 30.0, True, 0.07),
                                                       (37, 20.0, True, -0.05)])
def test_masks(window, softcap, sink, scale):
    check(48, [1, 9, 2], [600, 250, 0], window=window, softcap=softcap, scale=scale,
          head_sink=np.linspace(-1, 1, 48) if sink else None)


# The library's 64 MiB hold no segments of 64-row blocks: 16- and 32-row blocks (pa_latent.hip) on the
# same rows, in one chunk and in several
@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("H,new,past", [(16, [1, 1], [130, 2500]), (33, [1], [197]), (64, [1] * 3, [640] * 3),
                                        (128, [1, 2], [131, 1900]), (16, [5, 70], [60, 300])])
def test_smaller_blocks_in_the_static_workspace(H, new, past, dtype):
    check(H, new, past, dtype=dtype, static=True)


# contexts that keep the smaller blocks with any workspace
@pytest.mark.parametrize("H,past", [(16, [0, 31, 63, 95]), (16, [127] * 16), (64, [100 + i % 28 for i in range(32)])])
def test_short_contexts(H, past):
    check(H, [1] * len(past), past)
