"""Every way of calling the metadata operators gives the same result.

torch.ops.gaudirt.paged_attn(...) with positional metadata goes to the
registered operator without torch's argument search
(gaudirt_amd._call_directly); keyword calls, the overload, and calls under a
dispatch mode, a function mode or a trace take torch's own path.
"""

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_call_forms_agree():
    import torch
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    import gaudirt_amd

    gaudirt_amd.load_extension()
    op = torch.ops.gaudirt.paged_attn
    heads, kv_heads, d, rows, context = 8, 2, 128, 5, 64
    gen = torch.Generator(device="cuda").manual_seed(3)
    slots = rows * context
    mapping = torch.arange(slots, dtype=torch.int32).reshape(rows, context)
    positions = torch.tensor([0, 5, 31, 32, 63])
    requests = torch.arange(rows)
    meta = torch.classes.gaudirt.PagedMetadata(mapping[requests, positions].long(), requests, positions, mapping, slots)
    pool = gaudirt_amd.allocate_paged_kv(1, slots, kv_heads, d)
    pool.normal_(generator=gen)
    key_pool, value_pool = gaudirt_amd.kv_pool_views(pool, 0)
    q, k, v = (torch.randn(rows, n * d, generator=gen, device="cuda").to(torch.bfloat16)
               for n in (heads, kv_heads, kv_heads))
    scale = float(np.float32(1 / math.sqrt(d)))
    want = op(q, k, v, key_pool, value_pool, meta, d, scale)
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    calls = {
        "overload": lambda: op.default(q, k, v, key_pool, value_pool, meta, d, scale),
        "keywords": lambda: op(q, k, v, key_pool, value_pool, metadata=meta, head_dim=d, scale=scale),
        "options": lambda: op(q, k, v, key_pool, value_pool, meta, d, scale, softcap=0.0, sliding_window=-1),
        "trace": lambda: make_fx(lambda a, b, c: op(a, b, c, key_pool, value_pool, meta, d, scale))(q, k, v)(q, k, v),
        "compiled": lambda: torch.compile(lambda a, b, c: op(a, b, c, key_pool, value_pool, meta, d, scale),
                                          backend="eager")(q, k, v),
    }
    for name, call in calls.items():
        print(name, flush=True)
        assert torch.equal(call().view(torch.int16), want.view(torch.int16)), name
    for mode in (Dispatch, Function):
        seen.clear()
        with mode():
            got = op(q, k, v, key_pool, value_pool, meta, d, scale)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        assert any("paged_attn" in str(f) for f in seen), (mode, seen)
    with pytest.raises(RuntimeError, match="paged_attn"):
        op(q, k)
    with pytest.raises(RuntimeError, match="head dimension"):
        op(q, k, v, key_pool, value_pool, meta, 96, scale)
