"""The partial merge of the streaming decode at the edges of its split: sequences of one partial up
to several rounds of every workgroup size, all head sizes, one and several rows, against the oracle."""
import numpy as np
import pytest

import _oracle as orc
from pa_cases import make_case, run_gpu_op

pytestmark = pytest.mark.gpu


# (heads, kv_heads, head, block, past): one kv-head gives a lone sequence up to 1024 partials (four
# rounds of the widest merge), many sequences give few (the narrowest), the ragged ones both
MERGES = [
    (6, 1, 128, 16, [40000]), (4, 1, 64, 16, [33001]), (4, 2, 96, 32, [9000]),
    (8, 2, 256, 256, [16383]), (16, 1, 128, 16, [4097, 0, 31, 20000]),
    (8, 2, 128, 16, [500] * 11 + [7000]), (8, 4, 64, 16, [9 * i for i in range(70)]),
    (2, 2, 96, 16, [63, 64, 65, 2000] * 5),
    (64, 8, 96, 16, [40 * i for i in range(39)] + [6000]),  # many workgroups: whole rows of 96
]


@pytest.mark.parametrize("heads,kv,head,block,past", MERGES)
@pytest.mark.parametrize("dtype", [orc.BF16, orc.F16])
def test_merge_of_partials(heads, kv, head, block, past, dtype):
    max_blocks = max((p + 1 + block - 1) // block for p in past)
    case = make_case(heads, kv, head, len(past) * max_blocks, block, len(past), dtype=dtype,
                     seed=head + len(past), new_lens=[1] * len(past), past=past,
                     max_blocks=max_blocks, std=1.0)
    ref, ref_t, kc_ref, vc_ref = orc.paged_attention_op(case)
    out, kc, vc = run_gpu_op(case)
    assert np.array_equal(kc, kc_ref) and np.array_equal(vc, vc_ref)
    got, want = orc.decode(out, dtype), orc.decode(ref_t, dtype)
    # outputs rounded once to T: 2^-9 (bf16) / 2^-12 (fp16) of each value at most on either side
    assert orc.rel_l2(got, want) <= 2e-3
    rows = got.reshape(len(past), -1), want.reshape(len(past), -1)
    assert max(orc.rel_l2(a, b) for a, b in zip(*rows)) <= 4e-3
