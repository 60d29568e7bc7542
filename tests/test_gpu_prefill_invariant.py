"""Prefill chunks of paged_attn where their work list would be cut (one MI355X).

The list cuts row tiles along their keys by the work of the whole batch, so a
chunk's last bits depend on what runs beside it. In batch-invariant mode they
must not: the chunk alone, beside other chunks and in a plan made before the
mode was switched on gives the same bits. The same uncut list serves a call that
finds no memory for the partial results.
"""

import math

import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


class Layer:
    """One pool with four requests of up to 3000 tokens; chunk 0 is 100 rows at position 2500."""

    def __init__(self, heads, kv_heads, d):
        import torch

        import gaudirt_amd

        gaudirt_amd.load_extension()
        self.torch, self.heads, self.kv_heads, self.d, self.context = torch, heads, kv_heads, d, 3000
        gen = torch.Generator(device="cuda").manual_seed(heads + d)
        self.mapping = torch.randperm(4 * self.context // 4, generator=torch.Generator().manual_seed(1)).to(torch.int32)
        self.mapping = (self.mapping[:, None] * 4 + torch.arange(4, dtype=torch.int32)).reshape(4, self.context)
        self.slots = self.mapping.numel()
        self.pool = gaudirt_amd.allocate_paged_kv(1, self.slots, kv_heads, d)
        self.pool.normal_(generator=gen)
        self.pools = gaudirt_amd.kv_pool_views(self.pool, 0)

        def draw(n):
            return torch.randn(4, self.context, n * d, generator=gen, device="cuda").to(torch.bfloat16)

        self.q, self.k, self.v = draw(heads), draw(kv_heads), draw(kv_heads)

    def batch(self, chunks):
        """(metadata, query, key, value) of chunks (request, first position, rows)."""
        torch = self.torch
        requests = torch.cat([torch.full((n,), r) for r, _, n in chunks])
        positions = torch.cat([torch.arange(p, p + n) for _, p, n in chunks])
        meta = torch.classes.gaudirt.PagedMetadata(self.mapping[requests, positions].long(), requests, positions,
                                                   self.mapping, self.slots)
        at = (requests.cuda(), positions.cuda())
        return meta, self.q[at], self.k[at], self.v[at]

    def attend(self, batch):
        meta, q, k, v = batch
        out = self.torch.ops.gaudirt.paged_attn(q, k, v, *self.pools, meta, self.d, 1 / math.sqrt(self.d))
        return out.view(self.torch.int16)


CHUNK, OTHERS = (0, 2500, 100), [(1, 0, 40), (2, 1000, 64), (3, 2900, 90)]


@pytest.mark.parametrize("heads,kv_heads,d", [(32, 8, 128), (14, 2, 64), (16, 8, 256)])
def test_chunks_are_batch_invariant_in_batch_invariant_mode(heads, kv_heads, d):
    import gaudirt_amd
    from tests.test_prefill_schedule import build

    for chunks in ([CHUNK], [CHUNK, *OTHERS]):
        _, _, lst = build([n for _, _, n in chunks], [p for _, p, _ in chunks], heads=(heads, kv_heads, d),
                          capacity=1 << 16)
        assert lst.merge_count, "the list of these chunks is to be cut"
    layer = Layer(heads, kv_heads, d)
    alone, beside = layer.batch([CHUNK]), layer.batch([CHUNK, *OTHERS])
    cut = layer.attend(alone)  # this plan is older than the mode
    gaudirt_amd.set_batch_invariant_decode(True)
    try:
        want, got = layer.attend(alone), layer.attend(beside)[:CHUNK[2]]
        again = layer.attend(layer.batch([OTHERS[0], CHUNK]))[-CHUNK[2]:]
    finally:
        gaudirt_amd.set_batch_invariant_decode(False)
    torch = layer.torch
    assert torch.equal(got, want) and torch.equal(again, want)
    assert torch.equal(layer.attend(alone), cut)
    positions = np.arange(CHUNK[1], CHUNK[1] + CHUNK[2])
    problem = orc.Problem(alone[1].view(torch.int16).cpu().numpy().view(np.uint16),
                          layer.pool[0].view(torch.int16).cpu().numpy().view(np.uint16), np.zeros(CHUNK[2], np.int64),
                          positions, layer.mapping.numpy(), heads, kv_heads, d, float(np.float32(1 / math.sqrt(d))))
    reference = orc.direct_bf16_pv(problem)
    for out in (want, cut):
        orc.check_tolerance(out.cpu().numpy().view(np.uint16), reference, 2e-2, 2e-3)


def test_no_memory_for_the_partials():
    import torch

    import gaudirt_amd

    layer = Layer(32, 8, 128)
    batch = layer.batch([CHUNK])
    gaudirt_amd.set_batch_invariant_decode(True)
    want = layer.attend(batch)
    gaudirt_amd.set_batch_invariant_decode(False)
    cut = layer.attend(batch)
    assert not torch.equal(cut, want)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # Room for the output (1 MiB), not for 22 MiB of partials, which no free block holds either.
    limit = torch.cuda.memory_reserved() + (8 << 20)
    torch.cuda.set_per_process_memory_fraction(limit / torch.cuda.get_device_properties(0).total_memory)
    try:
        held = []
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 1000:
                held.append(torch.empty(21 << 20, dtype=torch.uint8, device="cuda"))
        got = layer.attend(batch)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)
    assert torch.equal(layer.attend(batch), cut)
