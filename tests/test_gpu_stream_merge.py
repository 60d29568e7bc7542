"""GPU parity of the balanced decode schedule's merge where few rows are spread over many workgroups.

Both merge forms (one wave per (row, head), eight waves up to 512 pairs), with
units of one part, of fewer parts than waves, of a number that does not divide
by the waves, and of over a hundred; against the CPU oracle, and bit for bit
between repeats.
"""

import numpy as np
import pytest

from oracle import oracle as orc
from tests import paged_cases as cases

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_ABS = 2e-2, 2e-3  # the flat gates of tests/test_gpu_decode_stream.py


@pytest.mark.parametrize("heads,kv_heads,d,lens", [
    (32, 8, 128, [9001]),                                  # about 128 parts a unit
    (14, 2, 64, [8000, 40]),                               # over 400 parts, and a unit of one
    (16, 8, 256, [5000, 100, 3]),
    (32, 8, 128, [5000] + [70] * 15),                      # 512 pairs: parts fewer than waves
    (32, 8, 128, [5000] + [70] * 16),                      # 544 pairs: one wave each
    (8, 1, 128, [2500] * 9),
])
def test_merge_of_many_parts(heads, kv_heads, d, lens):
    import torch
    from tests import gk_runner as runner

    case = cases.decode_case(len(lens) + d, len(lens), heads, kv_heads, d, 16,
                             sum((n + 15) // 16 for n in lens) + 1, lens)
    q, pool = runner.bf16_device(case.query), runner.bf16_device(case.pool)
    tables, d_lens = runner.to_device(case.block_tables), runner.to_device(case.lens)
    out = torch.full((len(lens), heads * d), float("nan"), dtype=torch.bfloat16, device="cuda")
    params = runner.decode_params(q, pool, tables, d_lens, heads, kv_heads, d, 16, case.scale, out)
    actual = None
    for _ in range(3):
        ws = runner.paged_decode(params)
        torch.cuda.synchronize()
        del ws
        assert actual is None or np.array_equal(runner.bits_of(out), actual)
        actual = runner.bits_of(out)
    assert np.isfinite(orc.bf16_to_f32(actual)).all()
    max_abs, mean_abs = orc.check_tolerance(actual, orc.direct_bf16_pv(case.oracle_problem()), MAX_ABS, MEAN_ABS)
    print(f"max_abs={max_abs:.3e} mean_abs={mean_abs:.3e}", flush=True)
