"""torch.compile of a function that calls a metadata operator (CPU: the call itself ends in torch's dispatch error).

The metadata is a script object that Dynamo cannot put into a graph, so it
breaks the graph there and calls the operator as eager code does. Nothing of
the operator's own Python call may be compiled in that.
"""

import warnings

import pytest


@pytest.mark.parametrize("name", ["paged_attn", "rotary_paged_attn", "rotary_embedding"])
def test_no_frame_of_the_operator_call_is_compiled(name):
    import torch

    import gaudirt_amd

    gaudirt_amd.load_extension()
    op = getattr(torch.ops.gaudirt, name)
    # Any real script object will do: the operator is not reached on the CPU.
    metadata = torch.ops.quantized.linear_prepack(
        torch.quantize_per_tensor(torch.ones(4, 4), 0.1, 0, torch.qint8), None)
    assert type(metadata) is torch.ScriptObject
    options = {"paged_attn": (128, 0.1), "rotary_paged_attn": (128, 128, True, 0.1),
               "rotary_embedding": (128, 128, True)}

    def layer(x, pool, m):
        x = x + 1
        tensors = {"paged_attn": (x, x, x, pool, pool), "rotary_paged_attn": (x, x, x, pool, pool, x),
                   "rotary_embedding": (x, x, x)}[name]
        return op(*tensors, m, *options[name])

    torch._dynamo.reset()
    torch._dynamo.utils.counters.clear()
    compiled = torch.compile(layer, backend="eager")
    with warnings.catch_warnings():
        warnings.simplefilter("error", UserWarning)
        for rows in (1, 2, 3):
            x = torch.zeros(rows, 256, dtype=torch.bfloat16)
            with pytest.raises((NotImplementedError, RuntimeError)):
                compiled(x, torch.zeros(1, 2, 128, dtype=torch.bfloat16), metadata)
    frames = torch._dynamo.utils.counters["frames"]
    assert frames["total"] and frames["total"] == frames["ok"], dict(frames)
    assert not torch._dynamo.utils.counters["unimplemented"]
