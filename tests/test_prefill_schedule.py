"""CPU test of the prefill work list (gaudirt_amd/csrc/prefill_schedule.hpp, the
code that gk_prefill_list_build runs): tests/prefill_schedule_test.cpp built with
g++, and the C entry's own checks (no GPU)."""

import ctypes
import pathlib
import subprocess

import numpy as np

from gaudirt_amd import capi

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_work_list_covers_every_step(tmp_path):
    exe = tmp_path / "prefill_schedule_test"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fsanitize=address,undefined", "-I",
                    str(ROOT / "gaudirt_amd" / "csrc"), str(ROOT / "tests" / "prefill_schedule_test.cpp"), "-o",
                    str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout + run.stderr
    assert run.stdout.strip() == "OK"


def build(rows, prefix, *, heads=(32, 8, 128), window=-1, capacity=4096, entry="gk_prefill_list_build"):
    lib, as_i32 = capi.load(), lambda a: np.ascontiguousarray(a, dtype=np.int32)
    rows, prefix = as_i32(rows), as_i32(prefix)
    first = as_i32(np.concatenate([[0], np.cumsum(rows)[:-1]]))
    words, lst = np.zeros(max(capacity, 1), dtype=np.int32), capi.PrefillList()
    ptr = lambda a: ctypes.c_void_p(a.ctypes.data)  # noqa: E731
    rc = getattr(lib, entry)(ptr(first), ptr(rows), ptr(prefix), len(rows), *heads, window, ptr(words), capacity,
                             ctypes.byref(lst))
    return rc, words, lst


def test_list_entry_checks():
    rc, _, lst = build([512], [15000], capacity=0)
    assert rc == capi.GK_ERR_WORKSPACE and lst.merge_count == 8 and lst.item_count > 8
    need = 8 * lst.item_count + 4 * lst.merge_count
    assert build([512], [15000], capacity=need - 1)[0] == capi.GK_ERR_WORKSPACE
    rc, words, lst = build([512], [15000], capacity=need)
    assert rc == capi.GK_OK
    assert (words[:8 * lst.item_count].reshape(-1, 8)[:, 4] > 0).all()
    assert build([8], [0], heads=(7, 2, 128))[0] == capi.GK_ERR_INVALID_ARGUMENT
    assert build([8], [0], heads=(8, 2, 96))[0] == capi.GK_ERR_INVALID_ARGUMENT
    assert build([-1], [0])[0] == capi.GK_ERR_INVALID_ARGUMENT
    # The launch checks the list, its workspace and the common parameters before anything is enqueued.
    lib, p = capi.load(), capi.PrefillParams()
    p.q_heads, p.kv_heads, p.head_dim, p.block_size, p.slots, p.scale = 32, 8, 128, 16, 1 << 15, 0.1
    p.q_row_stride = p.out_row_stride = 32 * 128
    for name in ("query", "pool", "block_tables", "out"):
        setattr(p, name, 256)
    lst.items = lst.merges = lst.row_request = 256
    size = lib.gk_prefill_list_workspace_bytes(ctypes.byref(p), ctypes.byref(lst))
    assert size == 8 * lst.part_slots * 256 * (128 + 2) * 4
    launch = lambda ws, n: lib.gk_paged_prefill_listed(ctypes.byref(p), ctypes.byref(lst), ws, n, None)  # noqa: E731
    assert launch(None, 0) == capi.GK_ERR_WORKSPACE
    assert launch(ctypes.c_void_p(256), size - 1) == capi.GK_ERR_WORKSPACE
    assert launch(ctypes.c_void_p(264), size) == capi.GK_ERR_WORKSPACE
    lst.row_request = None
    assert launch(ctypes.c_void_p(256), size) == capi.GK_ERR_INVALID_ARGUMENT
    lst.struct_size = 8
    assert launch(ctypes.c_void_p(256), size) == capi.GK_ERR_INVALID_ARGUMENT


def test_uncut_list_follows_each_sequence_alone():
    # 100 rows on a 2500-key prefix, alone and beside other chunks: the same two whole items.
    def items(rows, prefix):
        rc, words, lst = build(rows, prefix, entry="gk_prefill_list_build_uncut")
        assert rc == capi.GK_OK and lst.merge_count == 0 and lst.part_slots == 0
        return words[:8 * lst.item_count].reshape(-1, 8)

    alone = items([100], [2500])
    assert (alone[:, 5] == -1).all() and alone[:, 1].sum() == 100 and len(alone) == 2
    beside = items([100, 64, 90], [2500, 1000, 2900])
    assert {tuple(i) for i in alone} <= {tuple(i) for i in beside}
    assert build([100], [2500])[2].merge_count > 0
    assert build([100], [2500], capacity=8, entry="gk_prefill_list_build_uncut")[0] == capi.GK_ERR_WORKSPACE
