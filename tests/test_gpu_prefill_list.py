"""GPU parity of prefill over a work list (gk_paged_prefill_listed) against the CPU oracle.

Shapes whose items are cut along the keys, at the edges of the split: row tiles
with a remainder, pieces that end inside the causal diagonal, kv head counts
that divide the eight XCDs and ones that do not, every slot lookup (page of a
step, of a load, of a key), softcap, windows, and a call whose window is
narrower than its list's, so that whole pieces see no key.
"""

import ctypes

import numpy as np
import pytest

from oracle import oracle as orc
from tests import paged_cases as cases

pytestmark = pytest.mark.gpu

# The flat gates of tests/test_gpu_prefill.py: a merge adds fp32 roundings only.
MAX_ABS, MEAN_ABS = 2e-2, 2e-3


def run(case, list_window):
    import torch

    from gaudirt_amd import capi
    from tests import gk_runner as runner
    from tests.test_prefill_schedule import build

    rc, words, lst = build(case.chunks, case.prefixes, heads=(case.heads, case.kv_heads, case.head_dim),
                           window=list_window, capacity=1 << 16)
    assert rc == capi.GK_OK
    q, pool, tables = runner.bf16_device(case.query), runner.bf16_device(case.pool), runner.to_device(case.block_tables)
    out = torch.full((case.rows, case.heads * case.head_dim), float("nan"), dtype=torch.bfloat16, device="cuda")
    p = capi.PrefillParams()
    p.query, p.q_row_stride = q.data_ptr(), q.stride(0)
    p.pool, p.slots = pool.data_ptr(), pool.shape[2]
    p.block_tables, p.bt_stride, p.block_size = tables.data_ptr(), tables.stride(0), case.block_size
    p.q_heads, p.kv_heads, p.head_dim = case.heads, case.kv_heads, case.head_dim
    p.scale, p.softcap, p.sliding_window = case.scale, case.softcap, case.window
    p.out, p.out_row_stride = out.data_ptr(), out.stride(0)
    device_words, requests = runner.to_device(words), runner.to_device(case.requests.astype(np.int32))
    lst.items = device_words.data_ptr()
    lst.merges = device_words.data_ptr() + 4 * 8 * lst.item_count
    lst.row_request = requests.data_ptr()
    need = capi.load().gk_prefill_list_workspace_bytes(ctypes.byref(p), ctypes.byref(lst))
    # What an earlier call left in the workspace must not matter.
    ws = torch.full((need // 4 + 1,), float("nan"), device="cuda")
    capi.check(capi.load().gk_paged_prefill_listed(ctypes.byref(p), ctypes.byref(lst), ctypes.c_void_p(ws.data_ptr()),
                                                   need, capi.current_stream()))
    torch.cuda.synchronize()
    return runner.bits_of(out), lst


@pytest.mark.parametrize("heads,kv_heads,d,block,prefixes,chunks,softcap,window,list_window", [
    (32, 8, 128, 16, [1500], [70], 0.0, -1, -1),
    (32, 8, 128, 128, [900, 0, 2000, 64], [64, 9, 65, 200], 0.0, -1, -1),
    (24, 3, 128, 1, [3000], [33], 0.0, -1, -1),
    (14, 2, 64, 1, [1501], [37], 0.0, -1, -1),
    (14, 2, 64, 8, [700, 1300], [73, 36], 30.0, -1, -1),
    (32, 16, 64, 32, [2000], [129], 0.0, 1000, 1000),
    (16, 8, 256, 16, [1200], [65], 50.0, -1, -1),
    (16, 8, 256, 1, [777, 1500], [63, 8], 0.0, 700, 700),
    (128, 1, 128, 16, [2500], [5], 0.0, -1, -1),
    # The call's window is narrower than the list's: pieces without a key.
    (32, 8, 128, 16, [1500], [70], 0.0, 100, -1),
    (14, 2, 64, 1, [1501], [37], 0.0, 40, -1),
    (16, 8, 256, 16, [1200], [65], 50.0, 33, 600),
])
def test_split_items(heads, kv_heads, d, block, prefixes, chunks, softcap, window, list_window):
    case = cases.PrefillCase(heads + block + sum(chunks), heads, kv_heads, d, block, prefixes=prefixes, chunks=chunks,
                             softcap=softcap, window=window)
    if window > 0:  # slots that no row sees are poisoned, and their table entries gone
        used = np.zeros(case.slots, dtype=bool)
        tables = case.block_tables.copy()
        for s, (prefix, chunk) in enumerate(zip(case.prefixes, case.chunks)):
            first = max(0, int(prefix) - window + 1)
            for t in range(first, int(prefix + chunk)):
                used[case.block_tables[s, t // block] * block + t % block] = True
            tables[s, :first // block] = -1
        case.pool[:, :, ~used, :] = 0x7fc0
        problem = case.oracle_problem()
        case.block_tables = tables
    else:
        problem = case.oracle_problem()
    actual, lst = run(case, list_window)
    assert lst.merge_count > 0, "nothing was split"
    reference = orc.direct_bf16_pv(problem) if softcap == 0.0 and window < 0 else orc.fp32_softmax_attention(problem)
    assert np.isfinite(orc.bf16_to_f32(actual)).all()
    max_abs, mean_abs = orc.check_tolerance(actual, reference, MAX_ABS, MEAN_ABS)
    print(f"items={lst.item_count} merges={lst.merge_count} max_abs={max_abs:.3e} mean_abs={mean_abs:.3e}", flush=True)


@pytest.mark.parametrize("heads,kv_heads,d", [(16, 8, 256), (32, 8, 128), (14, 2, 64)])
def test_repeats_are_bit_identical(heads, kv_heads, d):
    # Every product of a step has to be complete before the step's maxima read
    # it: a maximum taken too early gives another base, and other last bits from
    # run to run.
    case = cases.PrefillCase(d, heads, kv_heads, d, 16, prefixes=[1500, 300], chunks=[300, 200])
    first, _ = run(case, -1)
    for _ in range(4):
        assert np.array_equal(run(case, -1)[0], first)
