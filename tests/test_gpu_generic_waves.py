"""The VALU attention kernel with 1, 4 and 16 wavefronts per row: key counts around its rounds (one
key, a round less one, whole rounds, a remainder), biases of -inf, all cache kinds of the fallback."""
import numpy as np
import pytest

import _oracle as orc
from pa_cases import make_case, run_gpu_op

pytestmark = pytest.mark.gpu


# fp32 sums in another order: 2^-24 sqrt(keys) of the row at most, far below 1e-5
@pytest.mark.parametrize("head", [64, 40, 256])
@pytest.mark.parametrize("past", [[0], [31], [126, 127, 128, 129], [300, 1], [2500],
                                  list(range(0, 700, 11))])
def test_fp32_decode(head, past):
    mb = max(p + 1 + 15 for p in past) // 16
    case = make_case(8, 2, head, len(past) * mb, 16, len(past), dtype=orc.F32, seed=head,
                     new_lens=[1] * len(past), past=past, max_blocks=mb, std=1.0)
    ref, ref_t, kc_ref, vc_ref = orc.paged_attention_op(case)
    out, kc, vc = run_gpu_op(case)
    assert np.array_equal(kc, kc_ref) and np.array_equal(vc, vc_ref)
    assert orc.rel_l2(out, ref_t) <= 1e-5


@pytest.mark.parametrize("new,past", [([16] * 40, [0] * 40), ([3], [13]), ([5, 90], [200, 0])])
def test_fp32_rows_with_window_softcap_and_sink(new, past):
    mb = max(n + p + 15 for n, p in zip(new, past)) // 16
    case = make_case(4, 4, 72, len(new) * mb, 16, len(new), dtype=orc.F32, seed=3, new_lens=new,
                     past=past, max_blocks=mb, std=1.0, window=40, softcap=5.0,
                     head_sink=[0.5, -1, 2, 0])
    out = run_gpu_op(case)[0]
    assert orc.rel_l2(out, orc.paged_attention_op(case)[1]) <= 1e-5


@pytest.mark.parametrize("head,cache", [(96, orc.I8), (200, orc.I4), (96, orc.E4M3)])
def test_coded_pages_off_the_matrix_cores(head, cache):
    case = make_case(6, 3, head, 60, 16, 2, dtype=orc.F16, cache_dtype=cache, seed=5,
                     new_lens=[1, 1], past=[400, 37], max_blocks=30, std=1.0)
    got, want = run_gpu_op(case)[0], orc.paged_attention_op(case)[1]
    assert orc.rel_l2(orc.decode(got, orc.F16), orc.decode(want, orc.F16)) <= 2e-3


@pytest.mark.parametrize("masked", [0, 1, 64, 150])
def test_bias_of_minus_infinity_hides_its_keys(masked):
    import torch
    import onnxruntime_ep_mlx_amd as ep
    g = torch.Generator(device="cuda").manual_seed(masked)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    q, k, v, pk, pv = rnd(1, 1, 512), rnd(1, 1, 128), rnd(1, 1, 128), *(rnd(1, 2, 180, 64)
                                                                       for _ in "kv")
    bias = torch.zeros((1, 1, 1, 161), device="cuda")
    bias[..., :masked] = -torch.inf
    out, nk, nv = ep.group_query_attention(
        q, k, v, pk, pv, torch.tensor([160], dtype=torch.int32, device="cuda"), 161,
        attention_bias=bias, num_heads=8, kv_num_heads=2)
    keys, vals = (t[0, :, masked:161].double().repeat_interleave(4, 0) for t in (nk, nv))
    p = torch.softmax((q.view(8, 1, 64).double() * keys).sum(-1) / 8.0, -1)
    want = (p[..., None] * vals).sum(1).reshape(1, 1, 512)
    assert ((out.double() - want).norm() / want.norm()).item() <= 1e-5
