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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,KV,hd", [(14, 2, 64), (28, 4, 128), (8, 2, 32)])
@pytest.mark.parametrize("keys", [130, 200, 256])
def test_uncut_decode_rows_are_as_exact_as_cut_ones(dtype, H, KV, hd, keys):
    """A narrow table, whose keys one block takes, and the same table with absent pages behind, whose keys are cut over blocks: the same sums in
    another order of 32-bit additions, so that few results round to another number."""
    from machserve_amd.kernels import get_ops
    ops, ps, S = get_ops(dtype, DEV), 64, 8
    got = []
    rows = [inputs(dtype, H, KV, hd, ps, keys - 1, 1, 7 * s + keys + hd) for s in range(S)]
    q, kp, vp = (torch.cat([r[i] for r in rows]) for i in range(3))
    pages = rows[0][3]
    table = torch.arange(S * pages, dtype=torch.int32, device=DEV).view(S, pages)
    for t in (table, torch.cat([table, table.new_full((S, 60), -1)], dim=1)):
        got.append(ops.decode_attention(q, kp, vp, t.contiguous(), i32([keys - 1] * S), H, KV, hd, ps, None, hd ** -0.5))
    tile = ops._attention_lib(hd)[4]
    cuts = [ops._decode_splits(S, KV, n, ps, None, tile, hd) for n in (pages, pages + 60)]
    assert cuts[0] == 1 and cuts[1] > 4, "the first is whole, a wave of the second has a tile at most"
    assert (got[0] != got[1]).float().mean().item() < 0.01
    assert error(got[0], torch.cat([r[4] for r in rows])) < {torch.bfloat16: 2.2e-3, torch.float16: 2.8e-4}[dtype]
