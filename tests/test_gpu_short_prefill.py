"""The planned image prefill of batches with fewer row blocks than workgroup slots: items in parts
with fp32 partials, against a float64 evaluation of every sequence."""
import numpy as np
import pytest

from test_gpu_mixed_batch import Mixed

pytestmark = pytest.mark.gpu

# heads, kv, head, block, new tokens, past: from the first batch the rule takes (96 items, 320 keys at
# head 64) and just below it to whole rounds of slots, one long item among short ones (16 parts), empty
# sequences, a single token and last row blocks of one row; at head 128 the grid launch keeps the first
SHAPES = [
    (32, 8, 128, 16, [384], [0]), (32, 8, 128, 16, [353], [0]), (32, 8, 128, 16, [320], [0]),
    (28, 4, 128, 16, [512], [2000]), (28, 4, 128, 32, [1500, 0, 1, 33], [0, 5, 300, 7]),
    (8, 1, 128, 16, [1601, 17], [0, 30000]), (64, 8, 64, 16, [250, 250], [1000, 4000]),
    (64, 8, 64, 256, [511], [0]), (8, 4, 96, 16, [2000, 700], [100, 2500]),
    (24, 4, 256, 16, [513], [700]), (24, 4, 256, 32, [100, 90, 110, 200], [3000, 0, 500, 129]),
    (32, 8, 128, 16, [500], [0]), (64, 8, 64, 16, [177], [143]), (64, 8, 64, 16, [176], [144]),
    # the longest item at the most keys that stay whole, and one more: 96 items of 734, 128 of 412
    (64, 8, 64, 16, [177], [557]), (64, 8, 64, 16, [177], [558]),
    (24, 4, 256, 16, [150] * 4, [262] * 4), (24, 4, 256, 16, [150] * 4, [263, 262, 150, 262]),
]
FORMS = [dict(rot=32), dict(dtype="float16", rot=32),
         dict(dtype="float16", window=700, softcap=20.0, sink=True), dict(window=130, sink=True)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
def test_short_prefill(shape, form):
    m = Mixed(*shape, **form)
    got = m.call()
    m.check(*got)
    again = m.call()
    assert all((a == b).all() for a, b in zip(got, again))  # whatever order the plan's atomics took
    bounded = m.call(validate=False, max_query_len=max(m.new),
                     max_context_len=max(n + p for n, p in zip(m.new, m.past)))
    m.check(*bounded)



@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
def test_grid_launch_of_the_same_batches(shape, form):
    """Without a bound on their contexts they run on the grid launch."""
    m = Mixed(*shape, **form)
    m.check(*m.call(validate=False, max_query_len=max(m.new)))


@pytest.mark.parametrize("dtype,most", [("bfloat16", 2.3e-3), ("float16", 2.9e-4)])
@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[3], SHAPES[6], SHAPES[9]])
def test_error_is_the_output_rounding(shape, dtype, most):
    """Two-part probabilities and fp32 partials leave the rounding of the output to T: an error
    uniform within half an ulp, whose rms is ulp / sqrt(12), at most 2^-7 / sqrt(12) = 2.26e-3 (bf16)
    or 2^-10 / sqrt(12) = 2.82e-4 (fp16) of values at the bottom of their binade, the worst case.
    fp16 at head 128 takes one-part probabilities on every prefill kernel: as much again for the
    rounding of the weights, independently."""
    import torch
    m = Mixed(*shape, dtype=dtype)
    out, k, v = m.call()
    H, kv = m.opts["num_heads"], m.opts["kv_num_heads"]
    d, g, n, past = m.q.shape[1] // H, H // kv, m.new[0], m.past[0]
    q = m.q[:n].double().view(n, kv, g, d)
    s = torch.einsum("nkgd,lkd->kgnl", q, m.rows(k, "k", 0, past + n)) * d ** -0.5
    s.masked_fill_(torch.arange(past + n, device="cuda")[None]
                   > past + torch.arange(n, device="cuda")[:, None], -np.inf)
    want = torch.einsum("kgnl,lkd->nkgd", torch.softmax(s, -1),
                        m.rows(v, "v", 0, past + n)).reshape(n, H * d)
    assert ((out[:n].double() - want).norm() / want.norm()).item() <= (
        most * 2 ** 0.5 if dtype == "float16" and d == 128 else most)


@pytest.mark.parametrize("heads,kv,head", [(32, 8, 128), (64, 8, 64), (16, 4, 96)])
def test_small_probabilities_of_large_values(heads, kv, head):
    """bf16 keeps its values' whole exponent range, and their weights need theirs: 64 keys of weight 1
    and values in [1, 2), then keys whose weights of 2^-26.5 meet values of 2^26 times as much.  The
    output is rounded to bf16 (2^-9 of it); hi + lo probabilities add 2^-16."""
    import torch
    n = 900 if head == 96 else 500
    m = Mixed(heads, kv, head, 16, [n], [0])
    m.q.zero_()
    m.q.view(n, heads, head)[..., 0] = 1.0
    k, v = m.k.view(n, kv, head), m.v.view(n, kv, head)
    k.zero_()
    k[64:, :, 0] = -26.5 * np.log(2.0) * head ** 0.5
    v.uniform_(1.0, 2.0, generator=torch.Generator(device="cuda").manual_seed(head))
    v[64:] *= 2.0 ** 26
    out = m.call()[0].double().view(n, kv, heads // kv, head)
    s = torch.einsum("lkd,d->kl", k.double(), m.q.view(n, heads, head)[0, 0].double()) * head ** -0.5
    w = s.exp()  # the same for every row: running sums give all of them
    want = (w.T[..., None] * v.double()).cumsum(0) / w.cumsum(1).T[..., None]
    err = ((out - want[:, :, None]).abs() / want[:, :, None]).amax().item()
    assert err <= 2.0 ** -8, err
