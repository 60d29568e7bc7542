"""GPU parity of short-context decode (one workgroup per unit, KV store included) against the CPU oracle.

The step is the reference's fused decode (src/bridge/paged_attention.cpp:66-76,
172-347): store the new rows, then attend. Run with what can go wrong in one
launch: rows that attend other rows' new keys, new slots that hold NaN before
the step, slots that are not stored, tiles with a remainder, every page size,
windows that start inside a page, query-head groups with padding or more than
one workgroup, the row counts around the store's limit, and lengths on both
sides of the rule that takes this path. The pool is compared bit for bit.
"""

import numpy as np
import pytest

from oracle import oracle as orc
from tests import paged_cases as cases

pytestmark = pytest.mark.gpu

# The flat gates of tests/test_gpu_decode.py: the same arithmetic per tile, summed by wave.
MAX_ABS, MEAN_ABS = 2e-2, 2e-3


@pytest.fixture(scope="module")
def runner():
    import torch
    assert torch.cuda.is_available()
    from tests import gk_runner
    return gk_runner


def step(runner, heads, kv_heads, d, block, lens, requests=None, softcap=0.0, window=-1, skip=(), seed=0,
         max_context=None, unit=True):
    """One decode step: row r attends lens[r] keys of requests[r], its own new key last. `unit`: one workgroup per
    unit has to be what the library takes, or must not be."""
    import torch

    from gaudirt_amd import capi

    rng = np.random.default_rng(seed + d + block + len(lens))
    lens = np.asarray(lens, dtype=np.int32)
    rows = len(lens)
    requests = np.arange(rows) if requests is None else np.asarray(requests)
    longest = np.array([max([int(n) for n, q in zip(lens, requests) if q == r] + [1]) for r in range(requests.max() + 1)])
    case = cases.decode_case(seed, len(longest), heads, kv_heads, d, block,
                             int(((longest + block - 1) // block).sum()) + 2, longest)
    positions = np.maximum(lens, 1) - 1
    slots = case.block_tables[requests, positions // block].astype(np.int64) * block + positions % block
    new_k, new_v = (cases.bf16_normal(rng, (rows, kv_heads * d)) for _ in range(2))
    query = cases.bf16_normal(rng, (rows, heads * d))
    stored = np.array([r for r in range(rows) if r not in skip], dtype=np.int64)
    before = case.pool.copy()
    before[:, :, slots[stored], :] = 0x7fc0  # what the new rows replace must not be read
    slots[list(skip)] = -1
    expected = before.copy()
    orc.kv_store(new_k[stored], new_v[stored], slots[stored], len(stored), expected, case.slots, kv_heads, d)

    q, pool, tables = runner.bf16_device(query), runner.bf16_device(before), runner.to_device(case.block_tables)
    d_lens, reqs, sm = (runner.to_device(a.astype(np.int32)) for a in (lens, requests, slots))
    k, v = runner.bf16_device(new_k), runner.bf16_device(new_v)
    out = torch.full((rows, heads * d), float("nan"), dtype=torch.bfloat16, device="cuda")
    params = runner.decode_params(q, pool, tables, d_lens, heads, kv_heads, d, block, case.scale, out, row_request=reqs,
                                  softcap=softcap, window=window, new_key=k, new_value=v, slot_mapping=sm,
                                  max_context=max_context)
    assert (runner.schedule_of(params) == capi.GK_DECODE_UNIT) == unit
    ws = runner.paged_decode(params)
    torch.cuda.synchronize()
    del ws
    assert np.array_equal(runner.bits_of(pool), expected), "KV store differs from the oracle"
    actual = runner.bits_of(out)
    assert np.isfinite(orc.bf16_to_f32(actual)).all()
    for _ in range(3):
        runner.paged_decode(params)
        torch.cuda.synchronize()
        assert np.array_equal(runner.bits_of(out), actual), "the same step twice gives other bits"
    mapping = orc.mapping_from_block_table(case.block_tables, block, int(longest.max()))
    live = np.flatnonzero(lens > 0)
    problem = orc.Problem(query[live], expected, requests[live], positions[live].astype(np.int64), mapping, heads,
                          kv_heads, d, case.scale, softcap, window)
    reference = orc.fp32_softmax_attention(problem) if softcap or window > 0 else orc.direct_bf16_pv(problem)
    max_abs, mean_abs = orc.check_tolerance(actual[live], reference, MAX_ABS, MEAN_ABS)
    assert (orc.bf16_to_f32(actual[lens <= 0]) == 0).all()
    print(f"max_abs={max_abs:.3e} mean_abs={mean_abs:.3e}", flush=True)


@pytest.mark.parametrize("heads,kv_heads,d", [(8, 2, 128), (14, 2, 64), (16, 8, 256), (4, 4, 128), (20, 1, 64),
                                              (40, 2, 128), (24, 8, 256)])
@pytest.mark.parametrize("block", [1, 4, 16, 128])
def test_geometries_and_pages(runner, heads, kv_heads, d, block):
    step(runner, heads, kv_heads, d, block, [1, 31, 32, 33, 255, 257, 500])


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("variant", ["window", "softcap", "both"])
def test_window_and_softcap(runner, d, variant):
    step(runner, 16, 4, d, 8, [1, 40, 70, 71, 300, 611], softcap=0.0 if variant == "window" else 30.0,
         window=-1 if variant == "softcap" else 70)


@pytest.mark.parametrize("block", [1, 16, 64])
def test_rows_attend_other_rows_new_keys(runner, block):
    # Rows of one request at successive positions (fewer than a prefill run),
    # out of order among other requests: each sees the new keys before its own.
    step(runner, 8, 2, 128, block, [100, 33, 101, 103, 64, 102, 34], requests=[0, 1, 0, 0, 2, 0, 1])


def test_rows_that_store_nothing_and_empty_rows(runner):
    step(runner, 8, 2, 128, 16, [100, 0, 65, 0, 31], skip=(1, 2, 3))


@pytest.mark.parametrize("rows", [1, 3, 8, 9, 64, 200, 256, 257])
def test_row_counts(runner, rows):
    # One kv head: up to 512 rows take this path; from 257 on the store is a launch of its own.
    rng = np.random.default_rng(rows)
    step(runner, 4, 1, 64, 1, rng.integers(1, 130, rows), seed=rows)


@pytest.mark.parametrize("d,few,many", [(64, 2048, 3072), (128, 1536, 2048), (256, 768, 1024)])
@pytest.mark.parametrize("block", [1, 32])
@pytest.mark.parametrize("above", [0, 1])
def test_lengths_around_the_rule(runner, d, few, many, block, above):
    # Fewer than 32 units and 32: each longest row on both sides of its limit.
    step(runner, 4, 1, d, block, [few + above, few - 33, 7], unit=not above)
    step(runner, 4, 1, d, block, [many + above, many - 33] + [5] * 30, unit=not above)


@pytest.mark.parametrize("heads,kv_heads,d,rows,longest", [
    (32, 8, 128, 33, 512), (32, 8, 128, 33, 513),      # four waves, then eight
    (32, 8, 128, 65, 128), (32, 8, 128, 65, 129),      # two waves, then four
    (8, 8, 128, 128, 512), (8, 8, 128, 128, 513),      # four waves, then the balanced schedule
    (8, 8, 128, 129, 100),                             # more units than the unit form takes
    (32, 8, 64, 65, 200), (32, 8, 64, 130, 128),
    (16, 8, 256, 33, 256), (16, 8, 256, 33, 257), (16, 8, 256, 65, 40),
])
@pytest.mark.parametrize("window", [-1, 60])
def test_many_units(runner, heads, kv_heads, d, rows, longest, window):
    rng = np.random.default_rng(rows + longest)
    unit = rows * kv_heads <= {64: 2048, 128: 1024, 256: 512}[d] and (longest, rows, window) != (513, 128, -1)
    step(runner, heads, kv_heads, d, 16, [longest, longest - 1] + list(rng.integers(0, 48, rows - 2)), window=window,
         skip=(2,), unit=unit)


def test_window_inside_a_page_at_the_limit(runner):
    # 2048 visible keys that start inside a page: one block-table entry more than keys / page.
    step(runner, 4, 1, 128, 16, [3001, 2500] + [9] * 30, window=2048)
    step(runner, 4, 1, 128, 1, [3001, 2500] + [9] * 30, window=2048)


def test_contexts_beyond_max_context(runner):
    # A graph replayed on rows that outgrew its max_context: more block-table
    # entries than the workgroup keeps in LDS.
    import torch

    case = cases.decode_case(5, 2, 4, 1, 128, 1, 6000, [2800, 100])
    q, pool = runner.bf16_device(case.query), runner.bf16_device(case.pool)
    tables, lens = runner.to_device(case.block_tables), runner.to_device(case.lens)
    out = torch.zeros(2, 4 * 128, dtype=torch.bfloat16, device="cuda")
    params = runner.decode_params(q, pool, tables, lens, 4, 1, 128, 1, case.scale, out, max_context=100)
    ws = runner.paged_decode(params)
    torch.cuda.synchronize()
    del ws
    orc.check_tolerance(runner.bits_of(out), orc.direct_bf16_pv(case.oracle_problem()), MAX_ABS, MEAN_ABS)


@pytest.mark.parametrize("heads,kv_heads,rows,longest,max_context", [
    (4, 1, 5, 2800, 100),      # eight waves: 2049 entries in LDS
    (32, 8, 34, 700, 300),     # four: 513
    (32, 8, 65, 300, 100),     # two: 257
])
@pytest.mark.parametrize("softcap", [0.0, 30.0])
@pytest.mark.parametrize("windowed", [False, True])
def test_steps_beyond_max_context(runner, heads, kv_heads, rows, longest, max_context, softcap, windowed):
    # The replayed step with its store: the entries that are read in place also
    # decide which keys are the new rows', whose slots hold NaN, and rows of one
    # request attend each other's. With a window that still needs more entries
    # than LDS holds.
    lens = [longest, longest - 1, longest - 2, 100, 7] + [1 + 3 * i % max_context for i in range(rows - 5)]
    requests = [0, 0, 0, 1, 2] + list(range(3, rows - 2))
    step(runner, heads, kv_heads, 128, 1, lens, requests=requests, softcap=softcap, skip=(4,), max_context=max_context,
         window=longest - 40 if windowed else -1)


def test_short_workspace_stays_refused(runner):
    """The workspace that the size query names has to be there although this path leaves it untouched."""
    import ctypes

    import torch
    from gaudirt_amd import capi

    case = cases.decode_case(3, 2, 8, 2, 128, 16, 16, np.array([40, 64]))
    q, pool, tables = runner.bf16_device(case.query), runner.bf16_device(case.pool), runner.to_device(case.block_tables)
    lens = runner.to_device(case.lens.astype(np.int32))
    out = torch.full((2, 8 * 128), 3.0, dtype=torch.bfloat16, device="cuda")
    params = runner.decode_params(q, pool, tables, lens, 8, 2, 128, 16, case.scale, out)
    lib = capi.load()
    need = lib.gk_paged_decode_workspace_bytes(ctypes.byref(params))
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    for pointer, size in ((ws.data_ptr(), need - 1), (None, need), (None, 0)):
        rc = lib.gk_paged_decode(ctypes.byref(params), ctypes.c_void_p(pointer), size, capi.current_stream())
        assert rc == capi.GK_ERR_WORKSPACE, (size, rc)
    torch.cuda.synchronize()
    assert (out == 3.0).all()
