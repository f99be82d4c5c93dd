"""Errors of the attention kernels against 64 bits, kernel against kernel: they round the same operands in the same places, so none may be further
off than the one it replaces."""
import math

import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu

i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731


def inputs(dtype, H, KV, hd, ps, before, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)  # noqa: E731
    pages = -(-(before + n) // ps)
    q, kp, vp = (2.0 * rnd(n, H * hd)).to(dtype), rnd(pages, KV, ps, hd), rnd(pages, KV, hd, ps)
    K = kp.permute(1, 0, 2, 3).reshape(KV, -1, hd)[:, :before + n].double().repeat_interleave(H // KV, 0)
    V = vp.permute(1, 0, 3, 2).reshape(KV, -1, hd)[:, :before + n].double().repeat_interleave(H // KV, 0)
    s = torch.matmul(q.double().view(n, H, hd).transpose(0, 1).contiguous(), K.transpose(1, 2).contiguous()) * hd ** -0.5
    see = torch.arange(before + n, device=DEV)[None] <= torch.arange(before, before + n, device=DEV)[:, None]
    want = torch.matmul(torch.softmax(s.masked_fill(~see, -math.inf), -1), V).transpose(0, 1).reshape(n, H * hd)
    return q, kp, vp, pages, want


def error(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,KV,hd", [(14, 2, 64), (28, 4, 128), (12, 2, 128), (8, 8, 64)])
@pytest.mark.parametrize("before,n", [(0, 200), (0, 700), (300, 128), (900, 64), (1500, 300), (3000, 64)])
def test_tiles_of_32_rows_are_no_further_off_than_the_general_kernel(dtype, H, KV, hd, before, n):
    from machserve_amd.kernels import get_ops
    ops, ps = get_ops(dtype, DEV), 64
    q, kp, vp, pages, want = inputs(dtype, H, KV, hd, ps, before, n, before + n + hd)
    rows = ops.attention_rows_per_block(hd)
    work = i32([(0, r) for r in range(0, n * (H // KV), rows)])
    run = lambda groups: ops.paged_attention(q, kp, vp, i32([list(range(pages))]), i32([0]), i32([n]), i32([before]), work, H, KV, hd, ps, None,  # noqa: E731
                                             hd ** -0.5, groups, 1)
    tiles, general = error(run(32), want), error(run(1), want)
    # 3 %: such comparisons differ by up to 1 %; where the exponentials refer to something up to 2^8 below a row's maximum it is 4 to 25 %.
    # Heads of 64 behind tables of 2,048 keys and more are left up to 2^6 behind (17 to 20 %).
    behind = hd == 64 and pages * ps >= 2048
    assert tiles <= (1.21 if behind else 1.03) * general, (tiles, general)
