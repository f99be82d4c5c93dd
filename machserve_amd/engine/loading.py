"""From a model folder (or a typed configuration plus tensors) to a model on the device
with its cache and step function."""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch

from ..cache import CacheManager, DeviceCache, pages_by_need
from ..config import load_config
from ..kernels import get_ops
from ..parts import DecoderModel, Runtime
from ..parts.base import Mixer
from ..weights import Checkpoint, TensorDict, load_weights
from .step import StepFunction

DTYPES = {"bfloat16": torch.bfloat16, "bf16": torch.bfloat16, "float16": torch.float16, "fp16": torch.float16,
          "f16": torch.float16, "half": torch.float16, "float32": torch.float32, "fp32": torch.float32, "f32": torch.float32}


def parse_dtype(name) -> torch.dtype:
    if isinstance(name, torch.dtype):
        if name in (torch.bfloat16, torch.float16, torch.float32):
            return name
    elif name in DTYPES:
        return DTYPES[name]
    raise ValueError(f"dtype {name!r}: choose bfloat16, float16 or float32")


@dataclass
class LoadedModel:
    config: object
    model: DecoderModel
    cache: CacheManager
    device_cache: DeviceCache
    step: StepFunction
    rt: Runtime


# The memory-side cache (256 MB) that every read from memory goes through.  A decode step reads all weights one after the other: what fits in it
# is still there a step later, and of more than it holds nothing is, because whatever comes later pushes out what came before.  So
# where the weights are more, the largest are read past it (the loads' non-temporal form, which leaves nothing there) and the smallest, up to this much, stay.
# A chain of products of eight rows, us each, through the cache and past it: 9,728 x 896 in 60 to 240 MB of weights 4.45 and 4.8 to 5.1, 300 MB 5.04 and 4.82,
# 400 to 2,000 MB 5.26 to 5.48 and 4.84; 11,264 x 2,048 8.2 and 9.4, 9.3 and 9.4, 10.4 and 9.5.
CACHED_WEIGHT_BYTES = 192 << 20


def mark_weights_past_cache(model: DecoderModel, kept: int = CACHED_WEIGHT_BYTES) -> int:
    """Marks the weights that steps of few rows read past the last-level cache (``past_cache`` on the tensor): none if all of them
    fit in ``kept`` bytes, else the largest, so that the others do.  Returns how many bytes are marked.  The mark changes the
    kind of load and no result; a view of a weight does not carry it."""
    found = {}
    again = {id(p) for i, b in enumerate(model.blocks) if model.order.count(i) > 1 for q in b.parts() for p in (q, *getattr(q, "sub_parts", lambda: [])())}
    for part in model.parts():
        if part is model.embedding and getattr(model.head, "weight", None) is not None:
            continue  # rows of a table: not read as a whole
        if id(part) in again:
            continue  # a layer that a step runs more than once finds its weights in the cache
        for value in vars(part).values():
            for t in value if isinstance(value, (list, tuple)) else (value,):
                if isinstance(t, torch.Tensor) and t.dim() >= 2 and t.dtype == model.rt.dtype:
                    found[t.data_ptr()] = t
    weights = sorted(found.values(), key=lambda t: t.numel())
    sizes = [t.numel() * t.element_size() for t in weights]
    fits = sum(sizes) <= kept
    marked = room = 0
    for t, size in zip(weights, sizes):
        t.past_cache = not fits and room + size > kept
        room += 0 if t.past_cache else size
        marked += size if t.past_cache else 0
    return marked


def mark_weights_ahead(model: DecoderModel) -> None:
    """Tells the mixers which weights come behind their attention: the matrices of the block's feed-forward, the smallest first (a long K under a
    narrow output gains most by it).  Only where the weights do not all stay in the last-level cache anyway."""
    if not hasattr(model.rt.ops, "AHEAD_BYTES"):
        return
    for block in model.blocks:
        part = getattr(block, "feed_forward", None)
        found = [t for t in vars(part).values() if isinstance(t, torch.Tensor) and t.dim() == 2 and t.dtype == model.rt.dtype] if part is not None else []
        for mixer in block.mixers():
            for m in (mixer, *getattr(mixer, "sub_parts", lambda: [])()):
                if isinstance(m, Mixer):
                    m.ahead = tuple(sorted(found, key=lambda t: t.numel())[:2])


def load_model(model_dir: Optional[str] = None, *, dtype="bfloat16", device: str = "cuda:0", page_size: int = 64,
               num_pages=None, max_tokens: Optional[int] = None, max_requests: int = 64,
               config=None, tensors=None, ops=None, use_graphs: bool = True, portion: Optional[int] = None) -> LoadedModel:
    """``model_dir`` holds config.json and model.safetensors; alternatively pass a typed
    ``config`` and a dict of ``tensors``.  Every group's pool has ``num_pages`` pages (a dict
    gives each group its own number), or enough for ``max_tokens`` tokens; with ``portion``
    (the most tokens of one request that a step will bring) a group of layers that see a window
    gets only what ``max_requests`` requests can hold of it at a time."""
    dt = parse_dtype(dtype)
    if config is None:
        config = load_config(model_dir)
    if ops is None:
        ops = get_ops(dt, device)
    rt = Runtime(torch.device(device), dt, ops)
    model = DecoderModel(config.to_spec(), rt)
    source = TensorDict(tensors) if tensors is not None else Checkpoint(model_dir)
    load_weights(model, source, rt)
    if mark_weights_past_cache(model) > 0:
        mark_weights_ahead(model)
    if num_pages is None:
        if max_tokens is None:
            max_tokens = 4096
        num_pages = (pages_by_need(max_tokens, max_requests, portion, page_size) if portion
                     else max(1, -(-max_tokens // page_size)))
    cache = CacheManager(model.cache_requests(), page_size, num_pages, max_requests)
    device_cache = DeviceCache(cache, dt, rt.device)
    model.bind_cache(device_cache)
    # the work lists of a step are cut in the unit that the attention kernels themselves report
    step = StepFunction(model, cache, rt, model.attention_rows_per_block() or 64, use_graphs)
    return LoadedModel(config, model, cache, device_cache, step, rt)
