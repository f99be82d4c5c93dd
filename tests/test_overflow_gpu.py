"""One request's overflow stays its own: values in the pages are finite whatever a request computes, so that neither a request that gets its
pages afterwards nor one that runs beside it can meet them (0 * inf and 0 * NaN are NaN)."""
import pytest
import torch

import befirax_util
import livovik_util
import melerax_util
import nubodra_util
import renanex_util
import salolorn_util
from gpu_util import DEV
from tiny_configs import TINY_A, TINY_B, TINY_C, random_prompt

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
HEADS_64 = dict(TINY_B, hidden_size=256, num_attention_heads=4, num_key_value_heads=2)
HEADS_128 = dict(TINY_B, hidden_size=512, num_attention_heads=4, num_key_value_heads=2)
CONFIGS = {"qwen2 16": TINY_A, "qwen2 32": TINY_B, "qwen2 48, windows": TINY_C, "qwen2 64": HEADS_64, "qwen2 128": HEADS_128}
for util in (befirax_util, livovik_util, melerax_util, nubodra_util, renanex_util, salolorn_util):
    CONFIGS.update({f"{util.__name__[:-5]} {name}": raw for name, raw in util.CONFIGS.items()})
ASTRAY = 3  # the token whose embedding is no number


def logits_of(lm, slot, tokens, prompt):
    from machserve_amd.engine import StepEntry
    out = [lm.step([StepEntry(slot, tokens[:prompt], list(range(prompt)))])]
    for t in tokens[prompt:]:
        out.append(lm.step([StepEntry(slot, [t], [0])]))
    return torch.cat(out).float()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_a_request_that_went_astray_leaves_nothing_to_others(name, dtype):
    from machserve_amd.config import config_from_dict
    from machserve_amd.engine import load_model
    from machserve_amd.weights import random_tensor_dict
    config = config_from_dict(dict(CONFIGS[name]))
    tensors = random_tensor_dict(config, 5, dtype, device=DEV)
    embed = "embed" if "embed" in tensors else "model.embed_tokens.weight"
    vocab = tensors[embed].shape[0]
    tokens = [t for t in random_prompt(80, vocab, 6) if t != ASTRAY][:41]
    got = []
    for left in ("nothing", "pages", "pages and a request"):
        own = dict(tensors)
        if left != "nothing":
            own[embed] = own[embed].clone()
            own[embed][ASTRAY] = float("nan")
        lm = load_model(config=config, tensors=own, dtype=dtype, device=DEV, page_size=16, num_pages=6, max_requests=2, use_graphs=False)
        if left != "nothing":
            other = lm.cache.admit()
            n = 91 if left == "pages" else 35
            logits_of(lm, other, [ASTRAY] * n, n - 3)
            assert all(bool(torch.isfinite(pool).all()) for pool in lm.cache.device.vpools.values()), "a value in the pages"
            if left == "pages":
                lm.cache.release(other)
        got.append(logits_of(lm, lm.cache.admit(), tokens, 35))
    keep = torch.arange(vocab, device=DEV) != ASTRAY  # (a head that shares the embedding has no such logit)
    assert bool(torch.isfinite(got[0]).all())
    for other in got[1:]:
        assert torch.equal(got[0][:, keep], other[:, keep])


@pytest.mark.parametrize("dtype", DTYPES)
def test_values_as_the_pages_hold_them(dtype):
    """The largest number in the place of an overflow, as it is otherwise."""
    from machserve_amd.kernels import get_ops
    ops, H, KV, hd, ps = get_ops(dtype, DEV), 2, 1, 64, 16
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    most = torch.finfo(dtype).max
    v = torch.tensor([float("inf"), float("-inf"), float("nan"), 3.0e38, -3.0e38, most, -most, 1.5, -0.0, 0.0] * 6 + [2.0, 1e-30, -1e-30, 7.0], device=DEV)
    qkv = torch.zeros(1, 1, (H + 2 * KV) * hd, device=DEV)
    qkv[0, 0, -hd:] = v
    want = v.nan_to_num(nan=-most, posinf=most, neginf=-most).clamp(-most, most).to(dtype)
    for how in ("rows", "decoded"):
        kp, vp = torch.zeros(2, KV, ps, hd, dtype=dtype, device=DEV), torch.zeros(2, KV, hd, ps, dtype=dtype, device=DEV)
        if how == "rows":
            ops.rope_kv_write(qkv, None, i32([0]), None, i32([ps + 5]), kp, vp, H, KV, hd, ps)
        else:
            ops.decode_attention_fused(qkv, torch.zeros(qkv.shape[-1], device=DEV), None, i32([ps]), kp, vp, i32([[1]]), i32([0]), H, KV, hd, ps, None, 0.125)
        assert torch.equal(vp[1, 0, :, 5 if how == "rows" else 0], want)
