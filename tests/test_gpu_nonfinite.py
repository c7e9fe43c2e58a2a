"""Infinities and NaNs in inputs reach the rows that see them, and no others: the VALU kernel's
rounds of several keys, and every merge of partial rows."""
import numpy as np
import pytest

import _oracle as orc
from pa_cases import make_case, make_latent_case, run_gpu_op

pytestmark = pytest.mark.gpu


# key counts that leave a wavefront's last round short, full and with one key over: rounds hold 8
# keys (2 beyond head 256) of each of 1, 4 or 16 wavefronts
@pytest.mark.parametrize("dtype,head", [(orc.F32, 64), (orc.F16, 40), (orc.F32, 96), (orc.F32, 200),
                                        (orc.F32, 320)])
@pytest.mark.parametrize("past", [[0, 1, 6, 7, 8, 14], [31, 62, 63, 64, 126, 127, 128, 300],
                                  list(range(0, 560, 7))])
def test_infinite_last_value_on_the_valu_kernel(dtype, head, past):
    mb = max(past) // 16 + 1
    case = make_case(8, 2, head, len(past) * mb, 16, len(past), dtype=dtype, seed=head + len(past),
                     new_lens=[1] * len(past), past=past, max_blocks=mb, std=1.0)
    want = orc.decode(orc.paged_attention_op(case)[1], dtype).reshape(-1, 8, head)
    value = orc.decode(case["value"], dtype).reshape(-1, 2, head)
    value[:, 0, 3], value[:, 1, 5] = np.inf, -np.inf
    case["value"] = orc.encode(value, dtype).reshape(-1, 2 * head)
    got = orc.decode(run_gpu_op(case)[0], dtype).reshape(-1, 8, head)
    assert (got[:, :4, 3] == np.inf).all() and (got[:, 4:, 5] == -np.inf).all()
    rest = np.ones(got.shape, bool)
    rest[:, :4, 3] = rest[:, 4:, 5] = False
    assert orc.rel_l2(got[rest], want[rest]) <= (1e-5 if dtype == orc.F32 else 2e-3)


def _nan_rows(case, hit, dtype):
    """hit: (token, query head) whose query is NaN; that output row is NaN, the others as they were."""
    H = case["num_heads"]
    want = orc.decode(run_gpu_op(case)[0], dtype)
    want = want.reshape(want.shape[0], H, -1)
    q = orc.decode(case["query"], dtype).reshape(want.shape[0], H, -1)
    for t, h in hit:
        q[t, h, 7] = np.nan
    got = orc.decode(run_gpu_op(dict(case, query=orc.encode(q, dtype).reshape(case["query"].shape)))[0],
                     dtype).reshape(want.shape)
    rest = np.ones(want.shape[:2], bool)
    for t, h in hit:
        assert np.isnan(got[t, h]).all(), (t, h)
        rest[t, h] = False
    np.testing.assert_array_equal(got[rest], want[rest])


# partial rows met by the decode merge (64, 256 and 1024 threads), the parts of a short prefill and
# the MLA blocks' merge (one and four groups)
@pytest.mark.parametrize("heads,kv,head,new,past", [
    (32, 8, 128, [1] * 64, [900 + 60 * i for i in range(64)]), (32, 8, 128, [1, 2], [3000, 700]),
    (24, 4, 256, [1], [9000]), (28, 4, 128, [512], [2000]), (8, 4, 96, [700, 800], [300, 2500])])
def test_nan_query_through_partial_rows(heads, kv, head, new, past):
    mb = max(n + p for n, p in zip(new, past)) // 32 + 1
    case = make_case(heads, kv, head, len(new) * mb, 32, len(new), dtype=orc.BF16, seed=head,
                     new_lens=new, past=past, max_blocks=mb, std=1.0)
    _nan_rows(case, [(0, 1), (sum(new) - 1, heads - 2)], orc.BF16)


@pytest.mark.parametrize("H,past", [(128, [6000, 4000]), (64, [2000 + 30 * i for i in range(40)])])
def test_nan_query_through_mla_partials(H, past):
    mb = max(past) // 16 + 1
    case = make_latent_case(H, 576, 512, len(past) * mb, 16, len(past), dtype=orc.BF16, seed=H,
                            new_lens=[1] * len(past), past=past, max_blocks=mb,
                            scale=192.0**-0.5, std=1.0)
    _nan_rows(case, [(0, 1), (len(past) - 1, H - 2)], orc.BF16)
