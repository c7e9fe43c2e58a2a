"""Infinities in inputs reach the rows that see them, and no others: the VALU kernel's rounds of
several keys."""
import numpy as np
import pytest

import _oracle as orc
from pa_cases import make_case, run_gpu_op

pytestmark = pytest.mark.gpu


# key counts that leave a wavefront's last round short, full and with one key over: rounds hold 8
# keys (2 beyond head 256) of each of 1, 4 or 16 wavefronts
@pytest.mark.parametrize("dtype,head", [(orc.F32, 64), (orc.F16, 40), (orc.F32, 320)])
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
