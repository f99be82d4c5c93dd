"""Products that norm their one row themselves, against the norm's own kernel and the product: the same numbers, and the stream with its pending sums; one to sixteen sums, one
to eight slices, tiles of 16 to 64 columns, rows of whole and partial kilobytes."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("N,K,P", [(1152, 896, 4), (1152, 896, 1), (512, 448, 3), (40, 384, 16), (2048, 1536, 5), (1000, 1024, 1), (7000, 576, 2), (200, 2112, 3)])
def test_a_product_that_norms_its_row(dtype, N, K, P):
    from machserve_amd.kernels import get_ops
    ops = get_ops(dtype, DEV)
    rnd = lambda s, seed, f=1.0: (torch.randn(s, generator=torch.Generator().manual_seed(seed)) * f).to(DEV)  # noqa: E731
    x, parts, nw, w = rnd((1, K), 1, 2.0), rnd((P, 1, K), 2), 1 + rnd((K,), 3, 0.1), rnd((N, K), 4, K ** -0.5).to(dtype)
    if dtype == torch.float32 and N * K > 1 << 20:  # (more slices, and so more blocks that would read the row)
        pytest.skip("in 32-bit not every size is taken")
    assert ops.norms_its_row(1, N, K, P, x, parts, w)
    old, plain_x = x.clone(), x.clone()
    plain = ops.linear_split(ops.rmsnorm(plain_x, nw, 1e-6, None, False, parts), w)
    for _ in range(2):
        out, x_new = ops.linear_split_row_normed(x, parts, nw, 1e-6, w)
        assert torch.equal(out, plain) and torch.equal(x_new, plain_x) and torch.equal(x, old)
        w.past_cache = True


def test_what_a_product_does_not_norm():
    from machserve_amd.kernels import KernelError, get_ops
    ops = get_ops(torch.bfloat16, DEV)
    f = lambda *s: torch.zeros(s, device=DEV)  # noqa: E731
    w = f(1152, 896).bfloat16()
    for M, N, K, P in [(2, 1152, 896, 4), (1, 1152, 896, 0), (1, 1152, 896, 17), (1, 4608, 3584, 4), (1, 1152, 904, 4), (1, 151936, 896, 4)]:
        assert ops._plan("ms_few_normed_takes", M, N, K, P) == 0
    odd = f(1 + 896)[1:].view(1, 896)
    assert not ops.norms_its_row(1, 1152, 896, 4, odd, f(4, 1, 896), w)
    with pytest.raises(KernelError):
        ops.linear_split_row_normed(odd, f(4, 1, 896), f(896), 1e-6, w)
    with pytest.raises(KernelError):
        ops.linear_split_row_normed(f(2, 896), f(4, 2, 896), f(896), 1e-6, w)
