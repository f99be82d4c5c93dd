"""Decode steps behind few keys: narrow block tables, whose attention is not cut, and the change to the wider tables as the request grows."""
import pytest
import torch

from gpu_util import DEV
from plain import qwen2_plain as P
from tiny_configs import TINY_A, random_prompt, read_for_plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_the_library_s_choice_of_decode_splits_behind_few_keys(dtype, hd):
    from machserve_amd.kernels import get_ops
    ops = get_ops(dtype, DEV)
    tile = ops._attention_lib(hd)[4]
    splits = lambda keys: ops._decode_splits(1, 2, keys // 16, 16, None, tile, hd)  # noqa: E731
    whole = dtype != torch.float32 and hd <= 128
    for tiles in (1, 4, 5, 8, 9, 16):
        assert splits(tiles * tile) == (1 if whole and tiles <= 8 else -(-tiles // 4))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("page", [16, 64, 128, 512])
def test_a_request_that_outgrows_the_narrow_table(tmp_path, page, dtype):
    """Tokens one by one across 256 keys, each position against the plain model."""
    from machserve_amd.engine import StepEntry, load_model
    from machserve_amd.weights import write_random_model
    d = write_random_model(dict(TINY_A, max_position_embeddings=512), 4, str(tmp_path / "short"))
    w, sizes = read_for_plain(d)
    toks = random_prompt(264, 512, 9)
    ww = w if dtype == torch.float32 else {k: v.to(torch.bfloat16).float() if v.dim() == 2 else v for k, v in w.items()}
    ref = P.forward(ww, sizes, toks)
    lm = load_model(d, dtype=dtype, device=DEV, page_size=page, num_pages=24)
    assert lm.step.short_pages == (256 // page if dtype != torch.float32 and page > 32 else 0)
    slot = lm.cache.admit()
    out = [lm.step([StepEntry(slot, toks[:246], list(range(246)))])]
    for t in toks[246:]:
        out.append(lm.step([StepEntry(slot, [t], [0])]))
    scale = ref.abs().max().item()
    allowed = 2e-5 + 2e-5 * scale if dtype == torch.float32 else 3e-2 * scale
    assert (torch.cat(out).float().cpu() - ref).abs().max().item() <= allowed
