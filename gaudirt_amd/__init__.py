"""MI355X-native paged-attention path of GaudiRT (gfx950 HIP kernels behind a C ABI).

Python view of the path, mirroring the reference's ``gaudirt`` operator API
for it (python/gaudirt/__init__.py, src/bridge/generic_private_use1.cpp:430-540):

- ``torch.ops.gaudirt.paged_attn`` / ``_paged_attn_validated`` /
  ``_advance_decode_lengths``, the rotary ops ``rotary_embedding`` /
  ``rotary_embedding_positions`` / ``_rotary_embedding_validated``, and
  ``torch.classes.gaudirt.PagedMetadata`` are registered by the HIP extension
  ``gaudirt_amd._C``, together with ``rotary_paged_attn`` (rotary embedding
  fused into the attention's KV store; no counterpart in the reference);
- ``allocate_paged_kv(layers, slots, kv_heads, head_dim)`` returns a zeroed
  head-major bf16 pool ``[layers, 2, kv_heads, slots, head_dim]`` from the
  stream-ordered block allocator, and ``kv_pool_views(pool, layer)`` its
  ``(key_pool, value_pool)`` views ``[slots, kv_heads, head_dim]``.

- ``set_batch_invariant_decode(enabled, partition_tokens=2048)``: decode rows
  of ``paged_attn`` on fixed split-K partitions, so each row's output is a
  function of that row alone, bit for bit (the reference's single-row replay,
  tests/paged_attention_smoke.py:145-150), and prefill chunks with their keys
  in one piece, so each chunk's output is a function of that chunk alone; off
  by default, where the schedules' split points depend on the whole batch. The
  environment variable ``GAUDIRT_AMD_BATCH_INVARIANT_DECODE`` (``1``, or a
  partition in keys) turns it on when the extension loads.

The extension is loaded on first use of any of these names (or by
``load_extension()``); a missing build raises ImportError. There is no other
implementation behind them.
"""

import os
import pathlib

_PACKAGE = pathlib.Path(__file__).resolve().parent
_ext = None

__all__ = ["load_extension", "PagedMetadata", "paged_attn", "allocate_paged_kv", "kv_pool_views",
           "advance_decode_lengths", "kv_allocator_stats", "paged_attn_kv_tile", "set_batch_invariant_decode",
           "batch_invariant_decode"]

# Keys per split-K partition of the batch-invariant decode mode.
BATCH_INVARIANT_PARTITION = 2048


def load_extension():
    """Import the HIP extension (registers torch.ops.gaudirt.* and the PagedMetadata class)."""
    global _ext
    if _ext is not None:
        return _ext
    import torch

    try:
        from . import _C  # noqa: F401
    except ImportError as exc:
        raise ImportError(
            "gaudirt_amd: the HIP extension _C is not built or cannot load; run `python -m gaudirt_amd.build` "
            f"({exc})") from exc
    from . import _C as ext
    _register_fakes(torch)
    _call_directly(torch)
    _ext = ext
    env = os.environ.get("GAUDIRT_AMD_BATCH_INVARIANT_DECODE", "").strip()
    if env and env != "0":
        set_batch_invariant_decode(True, BATCH_INVARIANT_PARTITION if env == "1" else int(env))
    return ext


def set_batch_invariant_decode(enabled=True, partition_tokens=BATCH_INVARIANT_PARTITION):
    """Decode rows of paged_attn on fixed partitions of `partition_tokens` keys (a
    multiple of 32 up to 8192) and prefill rows with their keys in one piece: every
    row's output then depends on its own sequence alone. Off: the library's
    schedules (the default; faster on skewed batches and on few prefill rows),
    whose split points follow the whole batch."""
    load_extension()._set_decode_partition(int(partition_tokens) if enabled else 0)


def batch_invariant_decode():
    """The fixed decode partition in keys, or 0 when the library chooses."""
    return load_extension()._decode_partition()


def _call_directly(torch):
    """Calls of the metadata operators without torch's per-call search for fake script objects.

    For an operator with a custom-class argument, ``torch.ops.gaudirt.op(...)``
    looks through all call arguments, as a tree, for the stand-ins that export
    and fake tracing use: 6 us of the 18.7 us that a small attention call took with it. These
    operators have exactly one such argument, the metadata; when it is the real
    object the search finds nothing and the registered operator is called next,
    which is all that happens here. Every other call (metadata by keyword, a
    stand-in, too few arguments) takes torch's own path, as do the overloads
    (``.default``) and all calls on a torch that keeps its operators elsewhere.

    Around such a call torch.compile breaks its graph. Torch's own call frames are
    then left alone; this one is marked so too, or Dynamo would try to compile it,
    fail on the operator and warn.
    """
    try:
        from torch._C._dynamo.eval_frame import _FrameAction, _FrameExecStrategy, set_code_exec_strategy
    except ImportError:
        return
    real = torch.ScriptObject

    def direct(base, position):
        class Direct(base):
            __slots__ = ()

            def __call__(self, /, *args, **kwargs):
                if len(args) > position and type(args[position]) is real:
                    return self._op(*args, **kwargs)
                return base.__call__(self, *args, **kwargs)

        set_code_exec_strategy(Direct.__call__.__code__, _FrameExecStrategy(_FrameAction.SKIP, _FrameAction.DEFAULT))
        Direct.__name__, Direct.__qualname__, Direct.__module__ = base.__name__, base.__qualname__, base.__module__
        return Direct

    for name, position in (("paged_attn", 5), ("rotary_paged_attn", 6), ("rotary_embedding", 3)):
        packet = getattr(torch.ops.gaudirt, name)
        if callable(getattr(packet, "_op", None)):
            packet.__class__ = direct(type(packet), position)


def _register_fakes(torch):
    """Meta kernels for torch.compile tracing (python/gaudirt/__init__.py:136-153)."""

    @torch.library.register_fake("gaudirt::paged_attn")
    def _fake_paged_attn(query, key, value, key_pool, value_pool, metadata, head_dim, scale, softcap=0.0,
                         sliding_window=-1):
        torch._check(key.shape[0] == query.shape[0])
        torch._check(value.shape[0] == query.shape[0])
        return torch.empty_like(query, memory_format=torch.contiguous_format)

    @torch.library.register_fake("gaudirt::_paged_attn_validated")
    def _fake_paged_attn_validated(query, key, value, key_pool, value_pool, locations, requests, positions,
                                   mapping, header, head_dim, scale, softcap=0.0, sliding_window=-1):
        torch._check(key.shape[0] == query.shape[0])
        torch._check(value.shape[0] == query.shape[0])
        torch._check(locations.shape[0] == query.shape[0])
        torch._check(requests.shape[0] == query.shape[0])
        torch._check(positions.shape[0] == query.shape[0])
        return torch.empty_like(query, memory_format=torch.contiguous_format)

    @torch.library.register_fake("gaudirt::_advance_decode_lengths")
    def _fake_advance_decode_lengths(seq_lens, orig_seq_lens):
        return torch.empty_like(seq_lens), torch.empty_like(orig_seq_lens)

    @torch.library.register_fake("gaudirt::rotary_embedding")
    def _fake_rotary_embedding(query, key, cache, metadata, head_dim, rotary_dim, is_neox):
        torch._check(key.shape[0] == query.shape[0])
        return (torch.empty_like(query, memory_format=torch.contiguous_format),
                torch.empty_like(key, memory_format=torch.contiguous_format))

    @torch.library.register_fake("gaudirt::rotary_embedding_positions")
    def _fake_rotary_embedding_positions(query, key, cache, positions, head_dim, rotary_dim, is_neox):
        torch._check(key.shape[0] == query.shape[0])
        torch._check(positions.shape[0] == query.shape[0])
        return (torch.empty_like(query, memory_format=torch.contiguous_format),
                torch.empty_like(key, memory_format=torch.contiguous_format))

    @torch.library.register_fake("gaudirt::_rotary_embedding_validated")
    def _fake_rotary_embedding_validated(query, key, cache, positions, header, context, head_dim, rotary_dim,
                                         is_neox):
        torch._check(key.shape[0] == query.shape[0])
        torch._check(positions.shape[0] == query.shape[0])
        return (torch.empty_like(query, memory_format=torch.contiguous_format),
                torch.empty_like(key, memory_format=torch.contiguous_format))

    @torch.library.register_fake("gaudirt::rotary_paged_attn")
    def _fake_rotary_paged_attn(query, key, value, key_pool, value_pool, cache, metadata, head_dim, rotary_dim,
                                is_neox, scale, softcap=0.0, sliding_window=-1):
        torch._check(key.shape[0] == query.shape[0])
        torch._check(value.shape[0] == query.shape[0])
        return torch.empty_like(query, memory_format=torch.contiguous_format)


def allocate_paged_kv(layers, slots, kv_heads, head_dim):
    return load_extension()._allocate_paged_kv(layers, slots, kv_heads, head_dim)


def kv_pool_views(pool, layer):
    """(key_pool, value_pool) of one layer: [slots, kv_heads, head_dim] views of the combined storage."""
    return pool[layer, 0].transpose(0, 1), pool[layer, 1].transpose(0, 1)


def kv_allocator_stats(device=0):
    return load_extension()._kv_allocator_stats(device)


def paged_attn_kv_tile(rows):
    return load_extension()._paged_attn_kv_tile(rows)


def __getattr__(name):
    if name in ("PagedMetadata", "paged_attn", "advance_decode_lengths"):
        load_extension()
        import torch

        return {
            "PagedMetadata": lambda: torch.classes.gaudirt.PagedMetadata,
            "paged_attn": lambda: torch.ops.gaudirt.paged_attn,
            "advance_decode_lengths": lambda: torch.ops.gaudirt._advance_decode_lengths,
        }[name]()
    raise AttributeError(f"module 'gaudirt_amd' has no attribute {name!r}")
