"""Products of few rows in 32-bit whose waves share out K, against 64 bits: steps of 32 numbers, waves with unequal numbers of them, one to sixteen slices, outputs that end
inside a tile, one and two tiles of rows; a row's sums are those of the row by itself."""
import pytest
import torch

from gpu_util import DEV, assert_close
from plain import qwen2_plain as P

pytestmark = pytest.mark.gpu
F32 = torch.float32


def rnd(shape, dtype, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype)


@pytest.mark.parametrize("M", [1, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(16, 384), (1000, 416), (200, 4160), (5632, 1024), (40, 16384), (20000, 576), (1152, 896)])
def test_products_in_32_bit_whose_waves_share_out_k(M, N, K):
    from machserve_amd.kernels import get_ops, interleave_gate_up
    ops = get_ops(F32, DEV)
    assert ops._few(M, N, K, True) and ops._few(M, N, K, False, True) and not ops._few(33, N, K, True) and not ops._few(M, N, 256, True)
    a, w, bias, x0 = rnd((M, K), F32, 1), rnd((N, K), F32, 2, K ** -0.5), rnd((N,), F32, 3), rnd((M, N), F32, 4)
    ref = P.linear(a.double(), w.double())
    ad, wd = a.to(DEV), w.to(DEV)
    parts = ops.linear_split(ad, wd)
    assert_close(parts.sum(0), ref, F32, "slices")
    assert_close(ops.linear(ad, wd, None, out_f32=True), ref, F32, "whole")
    assert_close(ops.linear(ad, wd, bias.to(DEV)), ref + bias.double(), F32, "with a bias")
    assert_close(ops.linear_act(ad, wd, "relu2"), torch.relu(ref) ** 2, F32, "activation")
    x = x0.to(DEV)
    pend = ops.linear_residual(ad, wd, x)
    assert_close(x.cpu() if pend is None else x.cpu() + pend.sum(0).cpu(), x0.double() + ref, F32, "into the stream")
    g, u = rnd((N // 2 + 3, K), F32, 5, 2 * K ** -0.5), rnd((N // 2 + 3, K), F32, 6, K ** -0.5)
    gated = P.silu(P.linear(a.double(), g.double())) * P.linear(a.double(), u.double())
    assert_close(ops.linear_swiglu(ad, interleave_gate_up(g, u).to(DEV), N // 2 + 3), gated, F32, "gated")
    alone = ops.linear_split(ad[M - 1:].contiguous(), wd)
    assert alone.shape[0] == parts.shape[0] and torch.equal(alone[:, 0], parts[:, M - 1])


@pytest.mark.parametrize("M", [1, 8, 20])
def test_a_pending_norm_in_32_bit_stands_alone_before_such_a_product(M):
    """Behind nothing pending, and behind sums: the norm's own kernel and the product, where both were one kernel."""
    from machserve_amd.config import NormSpec
    from machserve_amd.kernels import get_ops, interleave_gate_up
    from machserve_amd.parts import NORMS, ResidualStream, Runtime
    ops = get_ops(F32, DEV)
    K, N, I, eps = 896, 1152, 4864, 1e-6
    norm = NORMS.build(NormSpec("rmsnorm", K, eps), Runtime(torch.device(DEV), F32, ops))
    nw = 1 + rnd((K,), F32, 1, 0.1)
    norm.load({"weight": nw.to(DEV)})
    x, w, g, u = rnd((M, K), F32, 2, 2.0), rnd((N, K), F32, 3, K ** -0.5), rnd((I, K), F32, 4, K ** -0.5), rnd((I, K), F32, 5, K ** -0.5)
    a, wo = rnd((M, K), F32, 6), rnd((K, K), F32, 7, K ** -0.5)
    h = P.rms_norm(x, nw, eps).double()
    stream = ResidualStream(x.to(DEV).clone(), ops)
    assert_close(norm.pending(stream).linear_split(w.to(DEV)).sum(0), P.linear(h, w.double()), F32, "q/k/v")
    stream = ResidualStream(x.to(DEV).clone(), ops)
    stream.add_linear(a.to(DEV), wo.to(DEV))
    x2 = (x.double() + P.linear(a.double(), wo.double()))
    h = P.rms_norm(x2.float(), nw, eps).double()
    got = norm.pending(stream).linear_swiglu(interleave_gate_up(g, u).to(DEV), I)
    assert_close(got, P.silu(P.linear(h, g.double())) * P.linear(h, u.double()), F32, "gated")
    assert_close(stream.value(), x2, F32, "the stream itself")
