"""Into how many blocks the keys of rows behind long contexts are cut, heads of 64 in two-byte types: by the places of the chip (256 CUs)."""
import pytest
import torch

from gpu_util import DEV, assert_close

pytestmark = pytest.mark.gpu


def plan_of(dtype=torch.bfloat16):
    from machserve_amd.kernels import get_ops
    lib = get_ops(dtype, DEV)._attention_lib(64)[0]
    return lambda items, KV, T, pages: lib.ms_attention_splits_nd4(items, KV, T, 64, 64, pages, 0)


def test_splits_fill_the_chip_s_places():
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers are those of 256 CUs")
    plan = plan_of()
    # two blocks a CU (items x 2 KV heads x 2 blocks x splits <= 512), and three where a split keeps 1,664 keys
    assert plan(28, 2, 512, 133) == 4 and plan(28, 2, 512, 258) == 6
    assert plan(56, 2, 1024, 63) == 2 and plan(56, 2, 1024, 79) == 3 and plan(56, 2, 1024, 266) == 3
    assert plan(14, 2, 256, 254) == 9 and plan(14, 2, 256, 504) == 13
    # items that are more than half of the chip's places but no whole round
    assert plan(112, 2, 2048, 64) == 1, "no longer than twice the step's rows"
    assert plan(112, 2, 2048, 288) == 5 and plan(32, 8, 64, 126) == 3
    # a whole round and more
    assert plan(200, 2, 3600, 256) == 1 and plan(192, 2, 2048, 600) == 1


@pytest.mark.parametrize("items,KV,T,pages", [(28, 2, 512, 258), (56, 2, 1024, 266), (112, 2, 2048, 288), (32, 8, 64, 126), (3, 1, 70, 4000)])
def test_a_split_keeps_its_keys(items, KV, T, pages):
    n = plan_of()(items, KV, T, pages)
    assert 1 < n <= 64 and pages * 64 // n >= 1024


@pytest.mark.parametrize("before,n,H,KV", [(5100, 300, 14, 2), (6000, 2, 8, 8)])
def test_rows_behind_a_long_context(before, n, H, KV):
    """The library's own cut against uncut keys: the same attention."""
    from machserve_amd.kernels import get_ops
    ops, hd, ps = get_ops(torch.bfloat16, DEV), 64, 64
    g = torch.Generator(device=DEV).manual_seed(before)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    S = 3 if n > 2 else 32
    pages = -(-(before + n) // ps)
    q, kp, vp = rnd(S * n, H * hd), rnd(pages, KV, ps, hd), rnd(pages, KV, hd, ps)
    rows = ops.attention_rows_per_block(hd)
    work = i32([(s, r) for s in range(S) for r in range(0, n * (H // KV), rows)])
    run = lambda splits: ops.paged_attention(q, kp, vp, i32([list(range(pages))] * S), i32([s * n for s in range(S)]), i32([n] * S), i32([before] * S),  # noqa: E731
                                             work, H, KV, hd, ps, None, hd ** -0.5, 0, splits)
    assert_close(run(0), run(1), torch.bfloat16, "cut by the library")
