"""Each HIP kernel alone against its plain reference, at sizes other than the engine's:
head sizes in steps of 16, odd numbers of heads and groups, widths and vocabularies that
are no power of two, page sizes 16 to 128, single rows beside long portions."""
import math

import pytest
import torch

from emulated_ops import EmulatedOps
from gpu_util import DEV, assert_close
from plain import qwen2_plain as P

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def ops_for(dtype):
    from machserve_amd.kernels import get_ops
    return get_ops(dtype, DEV)


def rnd(shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,V,d", [(1, 50, 24), (37, 1000, 200), (300, 777, 896)])
def test_embed(dtype, T, V, d):
    ops = ops_for(dtype)
    table = rnd((V, d), dtype, 1)
    toks = torch.randint(0, V, (T,), generator=torch.Generator().manual_seed(2), dtype=torch.int32)
    got = ops.embed(toks.to(DEV), table.to(DEV))
    assert torch.equal(got.cpu(), table[toks.long()].float())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,d,eps", [(1, 8, 1e-6), (5, 200, 1e-5), (130, 896, 1e-6), (3, 5000, 1e-2), (7, 1536, 1e-6), (6, 4100, 1e-6)])
def test_rmsnorm(dtype, T, d, eps):
    ops = ops_for(dtype)
    x = rnd((T, d), torch.float32, 3, 3.0)
    w = 1 + rnd((d,), torch.float32, 4, 0.1)
    ref = P.rms_norm(x, w, eps)
    assert_close(ops.rmsnorm(x.to(DEV), w.to(DEV), eps), ref, dtype, "rmsnorm")
    rows = torch.tensor([T - 1, 0, T // 2], dtype=torch.int32)
    got = ops.rmsnorm(x.to(DEV), w.to(DEV), eps, rows.to(DEV), out_f32=True)
    assert_close(got, ref[rows.long()], torch.float32, "rmsnorm of gathered rows")
    # pending sums are folded in, and written back when no rows are gathered
    parts = rnd((3, T, d), torch.float32, 5)
    total = x + parts.sum(0)
    xd = x.to(DEV).clone()
    assert_close(ops.rmsnorm(xd, w.to(DEV), eps, partials=parts.to(DEV)), P.rms_norm(total, w, eps), dtype, "norm of sums")
    assert_close(xd, total, torch.float32, "sums written back")
    xd = x.to(DEV).clone()
    got = ops.rmsnorm(xd, w.to(DEV), eps, rows.to(DEV), True, parts.to(DEV))
    assert_close(got, P.rms_norm(total, w, eps)[rows.long()], torch.float32, "gathered norm of sums")
    assert torch.equal(xd.cpu(), x), "gathered rows leave the stream alone"
    ops.add_partials(xd, parts.to(DEV))
    assert_close(xd, total, torch.float32, "add_partials")
    # eight, nine, twelve and sixteen pending sums (more than eight come in a second round of loads), each
    # plane with a value of its own scale so that a plane left out or taken twice shows
    for n in (8, 9, 12, 16, 17):
        parts = torch.stack([rnd((T, d), torch.float32, 20 + k, 0.5 + 0.25 * k) for k in range(n)])
        total = x + parts.sum(0)
        xd = x.to(DEV).clone()
        assert_close(ops.rmsnorm(xd, w.to(DEV), eps, partials=parts.to(DEV)), P.rms_norm(total, w, eps), dtype, f"norm of {n} sums")
        assert_close(xd, total, torch.float32, f"{n} sums written back")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (7, 1000, 200), (64, 130, 896), (65, 257, 72), (300, 896, 4864),
                                   (129, 9728 + 16, 64),
                                   # the tiled kernel's K steps: one partial step, one whole, two whole, whole + partial
                                   (70, 100, 40), (130, 64, 64), (100, 96, 128), (513, 1200, 136), (2048, 1152, 904),
                                   # few tiles, whole K steps: four LDS buffers in turn, with four, five, seven and nineteen steps
                                   (64, 200, 256), (48, 264, 320), (40, 130, 448), (100, 72, 1216),
                                   # so many tiles that tiles of 128x160 save a round: whole tiles, and ragged rows and columns
                                   (1024, 9728, 136), (1000, 9700, 264),
                                   # tiles of 256x256 under eight waves, taken where they fill their rounds of a block a CU: whole
                                   # tiles with two whole K steps; ragged rows and columns with a partial last step; a long K
                                   (4096, 4096, 128), (4000, 4090, 136), (3840, 3584, 1600)])
def test_linear(dtype, M, N, K):
    ops = ops_for(dtype)
    a, w = rnd((M, K), dtype, 5), rnd((N, K), dtype, 6, K ** -0.5)
    b = rnd((N,), torch.float32, 7)
    ref = P.linear(a.double(), w.double(), b.double())
    assert_close(ops.linear(a.to(DEV), w.to(DEV), b.to(DEV), out_f32=True), ref, torch.float32 if dtype == torch.float32 else dtype, "linear f32 out")
    assert_close(ops.linear(a.to(DEV), w.to(DEV), None), P.linear(a.double(), w.double()), dtype, "linear")
    x = rnd((M, N), torch.float32, 8)
    xd = x.to(DEV).clone()
    # K cut over several blocks (a long K under few rows, or few tiles): partial sums; else added in the epilogue
    pending = ops.linear_residual(a.to(DEV), w.to(DEV), xd)
    if pending is not None:
        ops.add_partials(xd, pending)
    assert_close(xd, x.double() + P.linear(a.double(), w.double()), torch.float32 if dtype == torch.float32 else dtype, "linear_residual")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(65, 896, 4864), (300, 130, 1096), (2048, 896, 4864), (200, 200, 520), (100, 1536, 8960),
                                   (100, 1536, 1536), (130, 136, 264),
                                   # a very long K under few tiles of 256x256: K cut so that the slices fill the chip's round
                                   (1000, 3584, 16448)])
def test_linear_many_rows_cut_along_k(dtype, M, N, K):
    """A product with too few tiles to fill the chip is cut along K into ordered partial sums."""
    ops = ops_for(dtype)
    a, w = rnd((M, K), dtype, 41), rnd((N, K), dtype, 42, K ** -0.5)
    parts = ops.linear_split(a.to(DEV), w.to(DEV))
    if K >= 16384:
        assert parts.shape[0] == (1 if dtype == torch.float32 else 4), "56 tiles of 256x256 in four slices are a round of the chip"
    assert parts.shape[1:] == (M, N) and (dtype != torch.float32 or parts.shape[0] == 1)
    assert_close(parts.sum(0), P.linear(a.double(), w.double()), torch.float32 if dtype == torch.float32 else dtype)
    assert ops.linear_split(a.to(DEV), w.to(DEV), allow_partials=False).shape[0] == 1


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (3, 1000, 200), (8, 896, 4864), (17, 1152, 896), (17, 896, 904), (33, 130, 72),
                                   (64, 9728, 896), (5, 40000, 136), (48, 896, 896), (7, 1536, 1536), (3, 12000, 896)])
def test_linear_few_rows(dtype, M, N, K):
    """The weight-streaming kernels: partial sums that add up to the product, cut the same way
    for every number of rows, and a row's sums do not depend on the other rows."""
    ops = ops_for(dtype)
    a, w = rnd((M, K), dtype, 21), rnd((N, K), dtype, 22, K ** -0.5)
    ref = P.linear(a.double(), w.double())
    parts = ops.linear_split(a.to(DEV), w.to(DEV))
    assert parts.shape[1:] == (M, N)
    assert_close(parts.sum(0), ref, torch.float32 if dtype == torch.float32 else dtype, "sum of partial sums")
    whole = ops.linear_split(a.to(DEV), w.to(DEV), allow_partials=False)
    assert whole.shape == (1, M, N)
    assert_close(whole[0], ref, torch.float32 if dtype == torch.float32 else dtype, "one sum")
    assert_close(ops.linear(a.to(DEV), w.to(DEV), None, out_f32=True), ref, torch.float32 if dtype == torch.float32 else dtype)
    if M <= 32 and ops._tiled(M, N, K) == ops._tiled(1, N, K):
        # within one kernel family K is cut by N and K alone up to 32 rows: a row by itself gives the same bits
        alone = ops.linear_split(a[M - 1:].to(DEV).contiguous(), w.to(DEV))
        assert alone.shape[0] == parts.shape[0] and torch.equal(alone[:, 0], parts[:, M - 1])
    x0 = rnd((M, N), torch.float32, 23)
    x = x0.to(DEV)
    pend = ops.linear_residual(a.to(DEV), w.to(DEV), x)
    if pend is None:  # K inside one block, or a large weight under many rows (tiled kernel): added in the epilogue
        assert (parts.shape[0] == 1 and M <= 32) or ops._tiled(M, N, K)
        assert_close(x.cpu() - x0, ref, torch.float32 if dtype == torch.float32 else dtype, "added in place")
    else:
        assert torch.equal(pend, parts) and torch.equal(x.cpu(), x0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K,NP", [(1, 1152, 896, 0), (8, 1152, 896, 5), (16, 300, 264, 1), (3, 2048, 1536, 2),
                                      (5, 130, 1000, 3), (16, 4608, 3584, 6), (2, 64, 4864, 4)])
def test_products_with_the_norm_folded_in(dtype, M, N, K, NP):
    """rmsnorm(x + pending sums) times a weight in one kernel: the norm's factor applied to the
    finished sums, the stream with the sums added written to another buffer (the same bits as adding
    them in order), and the same with the gated activation."""
    from machserve_amd.kernels import interleave_gate_up
    ops = ops_for(dtype)
    # the engine folds the norm in only while there is little to read; the kernels take up to six pending sums
    # (never in half precision: the folded forms round x * weight before the division, which its range does not bear)
    assert ops.norm_folds_into(M, N, K, NP) == (dtype != torch.float16 and (NP == 0 or (NP == 1 and M <= 4)))
    assert not ops.norm_folds_into(17, N, K, 0)
    eps = 1e-5
    x = rnd((M, K), torch.float32, 31, 2.0)
    parts = rnd((NP, M, K), torch.float32, 32) if NP else None
    nw = 1 + rnd((K,), torch.float32, 33, 0.1)
    w = rnd((N, K), dtype, 34, K ** -0.5)
    total = x.clone()
    for p in range(NP):
        total += parts[p]
    h = P.rms_norm(total, nw, eps)
    ref = P.linear(h.double(), w.double())
    dev = lambda t: None if t is None else t.to(DEV)
    out, x_new = ops.linear_split_normed(dev(x), dev(parts), dev(nw), eps, dev(w))
    assert out.shape == (1, M, N) and (x_new is None) == (NP == 0)
    assert_close(out[0], ref, torch.float32 if dtype == torch.float32 else dtype, "product of the normed stream")
    if NP:
        assert torch.equal(x_new.cpu(), total), "the stream with its pending sums, added in order"
    I = N // 2 - 3
    g, u = rnd((I, K), dtype, 35, K ** -0.5 * 3), rnd((I, K), dtype, 36, K ** -0.5)
    ref = P.silu(P.linear(h.double(), g.double())) * P.linear(h.double(), u.double())
    got, x_new = ops.linear_swiglu_normed(dev(x), dev(parts), dev(nw), eps, interleave_gate_up(g, u).to(DEV), I)
    assert_close(got, ref, dtype, "gated product of the normed stream")
    if NP:
        assert torch.equal(x_new.cpu(), total)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K,I", [(8, 896, 896, 4864), (1, 896, 896, 4864), (20, 320, 264, 203), (32, 256, 128, 100),
                                     (5, 1000, 200, 50), (16, 1536, 904, 120), (3, 64, 72, 65536), (13, 2048, 136, 40),
                                     (17, 896, 896, 4864)])
def test_residual_product_prepares_the_norm_for_the_gated_product(dtype, M, N, K, I):
    """x += a w^T leaves x * norm_w and the rows' sums of squares beside the sum; the gated product of those rows
    divides its finished sums by the root mean square: together rmsnorm(x + a w^T) through gate and up."""
    from machserve_amd.kernels import interleave_gate_up
    ops = ops_for(dtype)
    if ops._plan("ms_skinny_prenorm_parts", M, N, K) < 1:
        pytest.skip("K is cut over several blocks for this shape, or the build is half precision (which rounds after the division)")
    eps = 1e-5
    a, w = rnd((M, K), dtype, 51), rnd((N, K), dtype, 52, K ** -0.5)
    x, nw = rnd((M, N), torch.float32, 53, 2.0), 1 + rnd((N,), torch.float32, 54, 0.1)
    x_new = x.double() + P.linear(a.double(), w.double())
    xd = x.to(DEV).clone()
    hn, ss = ops.linear_residual_prenorm(a.to(DEV), w.to(DEV), xd, nw.to(DEV))
    plain = torch.float32 if dtype == torch.float32 else dtype
    assert_close(xd, x_new, plain, "stream")
    assert_close(hn, xd.cpu().double() * nw.double(), dtype, "stream times the norm's weight")
    assert_close(ss.sum(0), (xd.cpu().double() ** 2).sum(1), torch.float32, "sums of squares")
    g, u = rnd((I, N), dtype, 55, N ** -0.5 * 3), rnd((I, N), dtype, 56, N ** -0.5)
    takes = ops.prenorm_swiglu_takes(M, N, K, 2 * ((I + 15) // 16) * 16)
    # the tiled form wants whole K steps of 64; at most 16 rows go to the few-rows form, which takes any K
    assert takes == (dtype == torch.bfloat16 and ((N % 64 == 0 and N >= 256) or M <= 16) and not ops._tiled(M, N, K))
    if takes:
        h = P.rms_norm(x_new.float(), nw, eps)
        ref = P.silu(P.linear(h.double(), g.double())) * P.linear(h.double(), u.double())
        got = ops.linear_swiglu_scaled(hn, ss, eps, interleave_gate_up(g, u).to(DEV), I)
        assert_close(got, ref, dtype, "gated product of the normed stream")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("scale,weight", [(1e4, 16.0), (1e-4, 0.02), (1.0, 1.0)])
@pytest.mark.parametrize("M", [1, 8, 16, 24])
def test_a_large_or_tiny_stream_goes_through_the_norm_and_its_reader(dtype, scale, weight, M):
    """The stream of a real checkpoint may be large (times a norm's weight: beyond half precision's 65,504) or tiny
    (among its subnormals): the norm's reader, whichever way it is run (the norm folded into the product, left to
    the product before it, or on its own), gives what the plain norm followed by the plain product gives, rounding
    after the division as the reference's f16 path does (crates/mach-model/src/kernels.rs:63-80)."""
    from machserve_amd.config import NormSpec
    from machserve_amd.kernels import interleave_gate_up
    from machserve_amd.parts import NORMS, ResidualStream, Runtime
    ops = ops_for(dtype)
    rt = Runtime(torch.device(DEV), dtype, ops)
    K, N, I, Ka, eps = 896, 1152, 4864, 896, 1e-13
    norm = NORMS.build(NormSpec("rmsnorm", K, eps), rt)
    nw = (1 + rnd((K,), torch.float32, 71, 0.1)) * weight
    norm.load({"weight": nw.to(DEV)})
    x = rnd((M, K), torch.float32, 72, scale)
    w = rnd((N, K), dtype, 73, K ** -0.5)
    g, u = rnd((I, K), dtype, 74, K ** -0.5 * 3 / weight), rnd((I, K), dtype, 75, K ** -0.5 / weight)
    a, wo = rnd((M, Ka), dtype, 76), rnd((K, Ka), dtype, 77, Ka ** -0.5 * scale)

    def rounded(h):
        return h.to(dtype).double()
    # 1. the norm's reader is a product that is summed later (q/k/v)
    stream = ResidualStream(x.to(DEV).clone(), ops)
    got = norm.pending(stream).linear_split(w.to(DEV)).sum(0)
    assert_close(got, P.linear(rounded(P.rms_norm(x, nw, eps)), w.double()), dtype, "q/k/v-like product of the normed stream")
    # 2. the reader is the gated product, and a product is still to be added to the stream before the norm
    stream = ResidualStream(x.to(DEV).clone(), ops)
    stream.add_linear(a.to(DEV), wo.to(DEV))
    got = norm.pending(stream).linear_swiglu(interleave_gate_up(g, u).to(DEV), I)
    x2 = (x.double() + P.linear(a.double(), wo.double())).float()
    h = rounded(P.rms_norm(x2, nw, eps))
    assert torch.isfinite(got.float()).all()
    assert_close(got, P.silu(P.linear(h, g.double())) * P.linear(h, u.double()), dtype, "gated product of the normed stream")
    assert_close(stream.value(), x2, torch.float32 if dtype == torch.float32 else dtype, "the stream itself")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,I,K", [(1, 4864, 896), (9, 168, 64), (16, 4864, 896), (200, 328, 192), (40, 1000, 576)])
def test_gated_products_with_another_activation(dtype, M, I, K):
    """The activation on the gate is an argument: the tanh form of GELU (crates/mach-model/src/kernels.rs:199-208)
    against the library's own, through every kernel that applies an activation: the tiled and the few-rows gated
    product, the one that applies the stream's norm itself, and the one that divides its finished sums."""
    import torch.nn.functional as F
    from machserve_amd.kernels import KernelError, interleave_gate_up
    ops = ops_for(dtype)
    gelu = lambda t: F.gelu(t, approximate="tanh")
    a, g, u = rnd((M, K), dtype, 9), rnd((I, K), dtype, 10, K ** -0.5), rnd((I, K), dtype, 11, K ** -0.5)
    gate, up = P.linear(a.double(), g.double()), P.linear(a.double(), u.double())
    ref = gelu(gate) * up
    assert (ref - P.silu(gate) * up).abs().max() > 0.03 * ref.abs().max(), "the test must tell the activations apart"
    w = interleave_gate_up(g, u).to(DEV)
    assert_close(ops.linear_swiglu(a.to(DEV), w, I, "gelu_tanh"), ref, dtype, "gated product, GELU")
    assert_close(ops.linear_swiglu(a.to(DEV), w, I, "silu"), P.silu(gate) * up, dtype, "gated product, SiLU by name")
    with pytest.raises(KernelError, match="gelu_erf"):
        ops.linear_swiglu(a.to(DEV), w, I, "gelu_erf")
    eps = 1e-5
    x, nw = rnd((M, K), torch.float32, 12, 2.0), 1 + rnd((K,), torch.float32, 13, 0.1)
    h = P.rms_norm(x, nw, eps).double()
    ref = gelu(P.linear(h, g.double())) * P.linear(h, u.double())
    if ops.norm_folds_into(M, w.shape[0], K, 0):
        got, _ = ops.linear_swiglu_normed(x.to(DEV), None, nw.to(DEV), eps, w, I, "gelu_tanh")
        assert_close(got, ref, dtype, "gated product of the normed stream, GELU")
    Ka = 72
    if ops.prenorm_swiglu_takes(M, K, Ka, w.shape[0]):
        b, wo = rnd((M, Ka), dtype, 14), rnd((K, Ka), dtype, 15, Ka ** -0.5)
        xd = x.to(DEV).clone()
        hn, ss = ops.linear_residual_prenorm(b.to(DEV), wo.to(DEV), xd, nw.to(DEV))
        h = P.rms_norm(xd.cpu(), nw, eps).double()
        ref = gelu(P.linear(h, g.double())) * P.linear(h, u.double())
        assert_close(ops.linear_swiglu_scaled(hn, ss, eps, w, I, "gelu_tanh"), ref, dtype, "gated product with row factors, GELU")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,I,K", [(1, 16, 8), (9, 160, 64), (70, 328, 192), (200, 4864, 896), (64, 4864, 896), (33, 264, 136),
                                   (64, 328, 256), (50, 1000, 576),
                                   # tiles of 128x160 (five pairs of gate and up tiles): whole, and ragged at both edges
                                   (2048, 4864, 896), (1000, 4850, 200),
                                   # tiles of 256x256 (two pairs of gate and up tiles a wave): whole, and ragged at both edges
                                   (4096, 2048, 128), (4000, 2040, 200),
                                   # the same tiles where they fill 0.89 of the chip under a short K
                                   (1536, 4864, 896)])
def test_linear_swiglu(dtype, M, I, K):
    from machserve_amd.kernels import interleave_gate_up
    ops = ops_for(dtype)
    a, g, u = rnd((M, K), dtype, 9), rnd((I, K), dtype, 10, K ** -0.5 * 3), rnd((I, K), dtype, 11, K ** -0.5)
    ref = P.silu(P.linear(a.double(), g.double())) * P.linear(a.double(), u.double())
    got = ops.linear_swiglu(a.to(DEV), interleave_gate_up(g, u).to(DEV), I)
    assert_close(got, ref, dtype, "swiglu")
    swapped = P.silu(P.linear(a.double(), u.double())) * P.linear(a.double(), g.double())
    assert (ref - swapped).abs().max() > 0.05 * ref.abs().max(), "the test must tell gate from up"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,KV,hd,ps,theta", [(4, 2, 16, 16, 1e4), (6, 1, 32, 32, 1e6), (5, 5, 48, 64, 5e4),
                                              (14, 2, 64, 64, 1e6), (3, 3, 128, 128, 1e6)])
def test_rope_kv_write(dtype, H, KV, hd, ps, theta):
    ops, emu = ops_for(dtype), EmulatedOps(dtype)
    T, pages = 45, 12
    qkv = rnd((T, (H + 2 * KV) * hd), torch.float32, 12)
    pos = torch.randint(0, 3000, (T,), generator=torch.Generator().manual_seed(13), dtype=torch.int32)
    perm = torch.randperm(pages * ps, generator=torch.Generator().manual_seed(14))[:T].to(torch.int32)
    j = torch.arange(hd // 2, dtype=torch.float32)
    inv = 1.0 / torch.pow(torch.tensor(theta, dtype=torch.float32), 2.0 * j / hd)
    kp, vp = torch.zeros(pages, KV, ps, hd, dtype=dtype), torch.zeros(pages, KV, hd, ps, dtype=dtype)
    q_ref = emu.rope_kv_write(qkv, None, pos, inv, perm, kp, vp, H, KV, hd, ps)
    # the emulation's rotation against the plain model's
    q_plain = P.rope(qkv[:, :H * hd].view(T, H, hd), pos, theta).reshape(T, H * hd)
    assert_close(q_ref, q_plain, dtype, "emulated rotation")
    kd, vd = torch.zeros_like(kp).to(DEV), torch.zeros_like(vp).to(DEV)
    q = ops.rope_kv_write(qkv.to(DEV), None, pos.to(DEV), inv.to(DEV), perm.to(DEV), kd, vd, H, KV, hd, ps)
    assert_close(q, q_plain, dtype, "q rotation")
    assert_close(kd, kp, dtype, "key pages")
    assert_close(vd, vp, dtype, "value pages")
    # without a table of frequencies nothing rotates
    q0 = ops.rope_kv_write(qkv.to(DEV), None, pos.to(DEV), None, None, None, None, H, KV, hd, ps)
    assert_close(q0, qkv[:, :H * hd], dtype, "no rotation")
    # three partial sums and a bias: the kernel adds them before it rotates
    parts = torch.stack([qkv * 0.5, qkv * 0.25 - 1.0, qkv * 0.25 + 1.0])
    bias = rnd(((H + 2 * KV) * hd,), torch.float32, 15)
    kp2, vp2 = torch.zeros_like(kp), torch.zeros_like(vp)
    q_ref2 = emu.rope_kv_write(qkv + bias, None, pos, inv, perm, kp2, vp2, H, KV, hd, ps)
    kd.zero_(), vd.zero_()
    q2 = ops.rope_kv_write(parts.to(DEV), bias.to(DEV), pos.to(DEV), inv.to(DEV), perm.to(DEV), kd, vd, H, KV, hd, ps)
    assert_close(q2, q_ref2, dtype, "q from partial sums")
    assert_close(kd, kp2, dtype, "key pages from partial sums")
    assert_close(vd, vp2, dtype, "value pages from partial sums")
    # seven and eleven partial sums (a portion of about a hundred rows cuts the projection's K seven times)
    for n in (7, 11):
        g = torch.Generator().manual_seed(16 + n)
        cut = torch.randn((n - 1, *qkv.shape), generator=g)
        parts = torch.cat([cut, (qkv - cut.sum(0)).unsqueeze(0)])
        kd.zero_(), vd.zero_()
        qn = ops.rope_kv_write(parts.to(DEV), bias.to(DEV), pos.to(DEV), inv.to(DEV), perm.to(DEV), kd, vd, H, KV, hd, ps)
        assert_close(qn, emu.rope_kv_write(parts.sum(0) + bias, None, pos, inv, perm, kp2.zero_(), vp2.zero_(), H, KV, hd, ps), dtype,
                     f"q from {n} partial sums")
        assert_close(kd, kp2, dtype, f"key pages from {n} partial sums")
        assert_close(vd, vp2, dtype, f"value pages from {n} partial sums")


def _dead_pages_removed(table, seqs, ps, window):
    """The block table as the cache manager hands it over once pages behind the window have been given
    back: a logical page that ends at or before ``cached - window + 1`` (no row of the step sees it) is -1."""
    table = table.clone()
    for i, (c, n) in enumerate(seqs):
        table[i, :max(0, c - window + 1) // ps] = -1
    return table


def _attention_case(dtype, H, KV, hd, ps, window, seqs, seed, peak=False, groups=0, splits=0, dead_pages=False):
    """seqs: list of (cached length, rows in this step).  Builds scattered pages holding random
    keys and values for positions < cached + rows and queries for the step's rows.  With
    ``dead_pages`` the kernel's block table has -1 where the pages lie wholly behind the window."""
    ops, emu = ops_for(dtype), EmulatedOps(dtype)
    g = H // KV
    gen = torch.Generator().manual_seed(seed)
    n_pages = sum(-(-(c + n) // ps) for c, n in seqs) + 3
    order = torch.randperm(n_pages, generator=gen).tolist()
    kp = rnd((n_pages, KV, ps, hd), dtype, seed + 1)
    vp = rnd((n_pages, KV, hd, ps), dtype, seed + 2)
    width = max(-(-(c + n) // ps) for c, n in seqs)
    table = torch.full((len(seqs), width), -1, dtype=torch.int32)
    q_start, q_len, pos0, work = [], [], [], []
    T = 0
    for i, (c, n) in enumerate(seqs):
        for p in range(-(-(c + n) // ps)):
            table[i, p] = order.pop()
        q_start.append(T), q_len.append(n), pos0.append(c)
        work += [(i, r0) for r0 in range(0, n * g, ops.attention_rows_per_block(hd))]
        T += n
    q = rnd((T, H * hd), dtype, seed + 3)
    if peak:
        # one far key stands out for one query row: scale that key and query so that the score
        # towers over the rest and a missed key shows in the output
        i, (c, n) = max(enumerate(seqs), key=lambda t: t[1][0])
        row, head, far = q_start[i] + n - 1, H - 1, (1 if not window else c + n - window)
        kvh = head // g
        page, off = int(table[i, far // ps]), far % ps
        qv = q[row, head * hd:(head + 1) * hd].float()
        kp[page, kvh, off, :] = (qv / qv.norm() * 8.0).to(dtype)
        q[row, head * hd:(head + 1) * hd] = (qv / qv.norm() * 8.0 * math.sqrt(hd) / 4).to(dtype)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    args = (i32(q_start), i32(q_len), i32(pos0), i32(work).view(-1, 2))
    if groups or splits:
        emu = EmulatedOps(torch.float32)  # the reference unrounded: the tolerance allows the output's one rounding
    emu.rows_per_block = ops.attention_rows_per_block(hd)
    ref = emu.paged_attention(q, kp, vp, table, *args, H, KV, hd, ps, window, hd ** -0.5)
    if dead_pages:
        table = _dead_pages_removed(table, seqs, ps, window)
        assert (table < 0).sum() > (table.shape[1] - torch.tensor([-(-(c + n) // ps) for c, n in seqs])).sum(), "no page is dead"
    got = ops.paged_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), table.to(DEV), *[a.to(DEV) for a in args], H, KV, hd,
                              ps, window, hd ** -0.5, groups, splits)
    return got, ref


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,KV,hd,ps", [(4, 2, 16, 16), (6, 1, 32, 32), (5, 5, 48, 16), (14, 2, 64, 64), (7, 7, 80, 32),
                                        (12, 2, 128, 64), (20, 1, 64, 128), (2, 1, 256, 16)])
def test_attention_mixed_batch(dtype, H, KV, hd, ps):
    seqs = [(0, 1), (0, 70), (130, 1), (37, 45), (ps - 1, 2), (ps, 1), (2 * ps - 1, 1)]
    got, ref = _attention_case(dtype, H, KV, hd, ps, None, seqs, 100 + hd)
    assert_close(got, ref, dtype, "attention")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("groups", [1, 2, 4])
@pytest.mark.parametrize("H,KV,hd,ps,window", [(4, 2, 16, 16, None), (14, 2, 64, 64, None), (6, 3, 128, 32, None),
                                               (2, 1, 256, 16, None), (6, 2, 64, 16, 100), (3, 1, 48, 32, 333)])
def test_attention_key_groups(dtype, groups, H, KV, hd, ps, window):
    """The keys of a block shared by 1, 2 or 4 groups of waves: short and long requests in one
    launch, lengths that end inside a round of tiles, and a far key that must not be missed."""
    seqs = [(0, 1), (0, 300), (517, 1), (700, 37), (3, 2), (1023, 1), (64 * groups, 1), (64 * groups - 1, 2)]
    got, ref = _attention_case(dtype, H, KV, hd, ps, window, seqs, 300 + hd + groups, peak=True, groups=groups)
    assert_close(got, ref, dtype, f"attention with {groups} key groups")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits,dead_pages", [(0, False), (3, False), (0, True)])
@pytest.mark.parametrize("H,KV,hd,ps,window", [(14, 2, 64, 64, None), (6, 2, 64, 16, 100), (20, 1, 64, 128, None), (8, 8, 64, 32, 333),
                                               (3, 1, 64, 16, 31)])
def test_attention_in_tiles_of_32_rows(dtype, splits, dead_pages, H, KV, hd, ps, window):
    """The kernel of 32-row tiles that the two-byte libraries have for a head size of 64 (blocks of 64 flat rows, two to a work
    item, two key groups, tiles loaded straight into two LDS stages, the block table in LDS; behind tables of 2,048 keys and more the
    reference maximum follows lazily), asked for by name: requests that end inside a tile, inside a round of two tiles and inside a block of
    rows, contexts of a few thousand keys, a window with the pages behind it given back, the keys cut over blocks, and
    a far key that must not be missed.  (The 32-bit library has no such kernel and answers with its general one.)"""
    if dead_pages and window is None:
        pytest.skip("pages are given back behind a window only")
    seqs = [(0, 1), (0, 300), (517, 1), (3000, 37), (3, 2), (1023, 1), (128, 1), (127, 2), (31, 2), (95, 130), (2040, 19)]
    got, ref = _attention_case(dtype, H, KV, hd, ps, window, seqs, 600 + ps + splits, peak=True, groups=32, splits=splits,
                               dead_pages=dead_pages)
    assert_close(got, ref, dtype, "attention in tiles of 32 rows")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits,dead_pages", [(0, False), (3, False), (0, True)])
@pytest.mark.parametrize("H,KV,ps,window", [(28, 4, 64, None), (6, 2, 16, 100), (20, 1, 128, None), (8, 8, 32, 333), (3, 1, 16, 31)])
def test_attention_in_tiles_of_32_rows_by_a_head_of_128(dtype, splits, dead_pages, H, KV, ps, window):
    """The same kernel for a head size of 128: one block to a work item, two blocks a CU, the reference always a row's maximum."""
    if dead_pages and window is None:
        pytest.skip("pages are given back behind a window only")
    seqs = [(0, 1), (0, 300), (517, 1), (3000, 37), (3, 2), (1023, 1), (128, 1), (127, 2), (31, 2), (95, 130), (2040, 19)]
    got, ref = _attention_case(dtype, H, KV, 128, ps, window, seqs, 650 + ps + splits, peak=True, groups=32, splits=splits, dead_pages=dead_pages)
    assert_close(got, ref, dtype, "attention in tiles of 32 rows, head size 128")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [64, 128])
def test_attention_reads_nothing_of_keys_that_are_not_there(dtype, hd):
    """Sixteen keys wholly beyond a request's rows or in pages given back are read from the start of the pool: what lies there stays out
    of the sums, in contexts that end in either half of a tile and windows that begin in either."""
    ops, g, KV, ps, window = ops_for(dtype), 3, 2, 16, 40
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    for pos0, n in [(0, 1), (0, 16), (0, 17), (31, 1), (32, 5), (63, 1), (64, 16), (100, 30)]:
        for w in (None, window):
            first = 0 if w is None else max(0, pos0 - w + 1) // ps
            pages = -(-(pos0 + n) // ps)
            kp, vp = rnd((pages + 1, KV, ps, hd), dtype, pos0), rnd((pages + 1, KV, hd, ps), dtype, pos0 + 1)
            q = rnd((n, KV * g * hd), dtype, pos0 + 2)
            table = torch.arange(1, pages + 1, dtype=torch.int32)
            table[:first] = -1
            rows = ops.attention_rows_per_block(hd)
            args = (table[None].to(DEV), i32([0]), i32([n]), i32([pos0]), i32([(0, r) for r in range(0, n * g, rows)]), KV * g, KV, hd, ps, w, hd ** -0.5)
            kp[0], vp[0] = 0, 0
            want = ops.paged_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), *args)
            kp[0], vp[0] = float("nan"), float("inf")
            got = ops.paged_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), *args)
            assert torch.equal(got, want) and bool(torch.isfinite(got).all()), (pos0, n, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("ps,window,splits", [(64, None, 1), (64, 50, 1), (64, None, 3), (16, 50, 1), (48, 50, 2)])
def test_keys_behind_a_narrow_block_table_are_read_from_the_pool(dtype, hd, ps, window, splits):
    """A table that holds none of the pages that a request's rows see: its keys are the pool's first page, and the requests beside it keep their results."""
    ops, g, KV = ops_for(dtype), 3, 2
    kp, vp = rnd((3, KV, ps, hd), dtype, 91).to(DEV), rnd((3, KV, hd, ps), dtype, 92).to(DEV)
    n0, n1 = ps - 3, 33
    q = rnd((n0 + n1, KV * g * hd), dtype, 93).to(DEV)
    rows = ops.attention_rows_per_block(hd)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    work = [[(i, r) for r in range(0, n * g, rows)] for i, n in ((0, n0), (1, n1))]
    tail = (KV * g, KV, hd, ps, window, hd ** -0.5, 32, splits)
    alone = ops.paged_attention(q[:n0].contiguous(), kp, vp, i32([[1]]), i32([0]), i32([n0]), i32([0]), i32(work[0]), *tail)
    both = ops.paged_attention(q, kp, vp, i32([[1], [2]]), i32([0, n0]), i32([n0, n1]), i32([0, 3000]), i32(work[0] + work[1]), *tail)
    assert torch.equal(both[:n0], alone)
    assert bool(torch.isfinite(both).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("ps", [16, 32, 48, 64, 96])
def test_prompts_of_any_page_size(dtype, hd, ps):
    """Prompts whose keys end before, at and behind a tile of 32 and a round of 64 keys, in pages that hold whole tiles and in pages that do not."""
    for window, seqs in ((None, [(0, 1), (0, 32), (0, 33), (31, 34), (60, 70), (100, 97)]), (50, [(0, 130), (90, 40), (64, 64)])):
        got, ref = _attention_case(dtype, 4, 2, hd, ps, window, seqs, 300 + ps, groups=32)
        assert_close(got, ref, dtype, f"window {window}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits", [2, 5, 64])
@pytest.mark.parametrize("H,KV,hd,ps,window", [(4, 2, 16, 16, None), (14, 2, 64, 64, None), (6, 3, 128, 32, None),
                                               (6, 2, 64, 16, 100), (3, 1, 48, 32, 333)])
def test_attention_key_splits(dtype, splits, H, KV, hd, ps, window):
    """The keys of a block of rows cut over several blocks and merged: short and long requests in
    one launch (most splits of the short ones are empty), and a far key that must not be missed."""
    seqs = [(0, 1), (0, 300), (517, 1), (1500, 37), (3, 2), (1023, 1), (128, 1), (127, 2)]
    got, ref = _attention_case(dtype, H, KV, hd, ps, window, seqs, 400 + hd + splits, peak=True, splits=splits)
    assert_close(got, ref, dtype, f"attention with the keys cut over {splits} blocks")


def test_the_library_s_choice_of_key_splits():
    """How many blocks share the keys of a block of rows when the caller leaves it to the library: none for block
    tables that may belong to prompts running whole (no wider than twice the step's rows) and for a full chip; few rows
    behind a long context are cut, in the kernel of 32-row tiles (head size 64, two-byte elements) so that blocks times
    splits stay within the chip's CUs, at least 1,024 keys a split; a window bounds the keys that count."""
    ops = ops_for(torch.bfloat16)
    lib = ops._attention_lib(64)[0]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    plan = lambda n_work, KV, T, hd, ps, width, window: lib.ms_attention_splits_nd4(n_work, KV, T, hd, ps, width, window)
    assert plan(56, 2, 1024, 64, 64, 32, 0) == 1                     # a prompt of 1,024 tokens whole
    assert plan(84, 2, 1536, 64, 64, 32, 0) == 1
    assert plan(14, 2, 256, 64, 64, 256, 0) == min(cus // 28, 16)    # 256 rows behind thousands of keys
    assert plan(28, 2, 512, 64, 64, 128, 0) == min(cus // 56, 8)
    assert plan(56, 2, 1024, 64, 64, 64, 0) == min(cus // 112, 4)
    assert plan(200, 2, 3600, 64, 64, 256, 0) == 1                   # the chip is full
    assert plan(1, 2, 1, 64, 64, 4096, 0) == 64                      # never more than the kernels take
    assert plan(14, 2, 256, 64, 64, 256, 500) == 1                   # a window of 500 keys: nothing to cut
    assert plan(4, 2, 64, 64, 16, 64, 0) == min(-(-384 // 8), 1024 // 512)   # a short table: the general kernel's rule
    lib128 = ops._attention_lib(128)[0]
    assert lib128.ms_attention_splits_nd8(7, 4, 256, 128, 64, 128, 0) == min(-(-384 // 28), 8192 // 512)
    f32 = ops_for(torch.float32)._attention_lib(64)[0]
    assert f32.ms_attention_splits_nd4(14, 2, 256, 64, 64, 256, 0) == min(-(-384 // 28), 16384 // 512)   # no 32-row kernel in 32-bit


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 17, 64, 100])
def test_attention_window(dtype, window):
    seqs = [(0, 150), (200, 1), (63, 3), (0, 1)]
    got, ref = _attention_case(dtype, 6, 2, 32, 16, window, seqs, 200 + window)
    assert_close(got, ref, dtype, f"attention with window {window}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window,splits", [(17, 0), (100, 0), (100, 3), (333, 0)])
def test_attention_window_with_pages_given_back(dtype, window, splits):
    """The pages behind the window are gone (-1 in the block table), as the cache manager leaves them:
    the kernel never looks a dead page up, whichever key tile, group of waves or split would hold it; the far
    key at the window's edge still counts."""
    seqs = [(0, 150), (200, 1), (63, 3), (0, 1), (700, 30), (1023, 1)]
    got, ref = _attention_case(dtype, 6, 2, 32, 16, window, seqs, 500 + window, peak=True, splits=splits, dead_pages=True)
    assert_close(got, ref, dtype, f"attention with window {window} and dead pages")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [None, 300])
def test_attention_far_key_stands_out(dtype, window):
    seqs = [(700, 1), (0, 5), (400, 40)]
    got, ref = _attention_case(dtype, 8, 2, 64, 64, window, seqs, 300, peak=True)
    assert_close(got, ref, dtype, "attention with a far key that dominates")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,KV,hd,ps,window", [(4, 2, 16, 16, None), (6, 1, 32, 32, None), (5, 5, 48, 16, 40),
                                               (14, 2, 64, 64, None), (16, 1, 80, 32, 100), (12, 2, 128, 64, None),
                                               (2, 1, 256, 16, None), (14, 2, 64, 64, 1)])
def test_decode_attention(dtype, H, KV, hd, ps, window):
    """One row per request, contexts from 0 to a few thousand keys, scattered pages; against the
    plain attention of the same rows, and against the general kernel."""
    ops, emu = ops_for(dtype), EmulatedOps(dtype)
    lens = [0, 1, ps - 1, ps, 130, 700, 2049] if hd < 256 else [0, 5, 300]
    gen = torch.Generator().manual_seed(500 + hd)
    n_pages = sum(-(-(c + 1) // ps) for c in lens) + 2
    order = torch.randperm(n_pages, generator=gen).tolist()
    kp, vp = rnd((n_pages, KV, ps, hd), dtype, 501), rnd((n_pages, KV, hd, ps), dtype, 502)
    width = max(-(-(c + 1) // ps) for c in lens)
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    for i, c in enumerate(lens):
        for p in range(-(-(c + 1) // ps)):
            table[i, p] = order.pop()
    S = len(lens)
    q = rnd((S, H * hd), dtype, 503)
    # one far key towers over the rest for the longest request's last head
    c = lens[-1]
    far = 3 if not window else max(0, c - window + 1)
    qv = q[S - 1, (H - 1) * hd:].float()
    kp[int(table[S - 1, far // ps]), KV - 1, far % ps, :] = (qv / qv.norm() * 8.0).to(dtype)
    q[S - 1, (H - 1) * hd:] = (qv / qv.norm() * 8.0 * math.sqrt(hd) / 4).to(dtype)
    pos0 = torch.tensor(lens, dtype=torch.int32)
    ref = emu.decode_attention(q, kp, vp, table, pos0, H, KV, hd, ps, window, hd ** -0.5)
    got = ops.decode_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), table.to(DEV), pos0.to(DEV), H, KV, hd, ps, window, hd ** -0.5)
    assert_close(got, ref, dtype, "decode attention")
    ar = torch.arange(S, dtype=torch.int32)
    work = torch.stack([ar, torch.zeros_like(ar)], 1).contiguous()
    gen_out = ops.paged_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), table.to(DEV), ar.to(DEV), torch.ones_like(ar).to(DEV),
                                  pos0.to(DEV), work.to(DEV), H, KV, hd, ps, window, hd ** -0.5)
    assert_close(got, gen_out.float().cpu(), dtype, "decode kernel against the general kernel")
    # a request alone (other split count) agrees within rounding
    one = ops.decode_attention(q[S - 1:].to(DEV).contiguous(), kp.to(DEV), vp.to(DEV), table[S - 1:].to(DEV).contiguous(),
                               pos0[S - 1:].to(DEV), H, KV, hd, ps, window, hd ** -0.5)
    assert_close(one, ref[S - 1:], dtype, "decode attention of one request")
    if window:
        # the pages behind the window given back, as the cache manager leaves the table
        dead = _dead_pages_removed(table, [(c, 1) for c in lens], ps, window)
        assert (dead[S - 1] < 0).sum() > 0
        got = ops.decode_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), dead.to(DEV), pos0.to(DEV), H, KV, hd, ps, window, hd ** -0.5)
        assert_close(got, ref, dtype, "decode attention with dead pages")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,KV,hd,ps,window,P_", [(4, 2, 16, 16, None, 1), (6, 1, 32, 32, None, 3), (5, 5, 48, 16, 40, 1),
                                                  (14, 2, 64, 64, None, 2), (12, 2, 128, 64, None, 1), (16, 1, 80, 32, 100, 1)])
def test_decode_attention_fused(dtype, H, KV, hd, ps, window, P_):
    """Bias, rotation, cache write and attention from partial sums of the projection; twice in a
    row with the same pages, the second time one position on, as decoding does."""
    _fused_decode_attention(dtype, H, KV, hd, ps, window, P_, [0, 1, ps - 1, ps, 130, 700, 2049, 63, 64])


# Three sums to more than the eight that are asked for first, heads of up to 64 and above; keys cut over blocks and (`short`) not, where requests have no key but the row's own,
# keys for some of the four waves and for all.  28 heads over 4 of 128 and 16 over 1 of 80 are 1,152 and 1,440 columns: those that a thread asks for first, and more behind them.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("short", [False, True])
@pytest.mark.parametrize("H,KV,hd,ps,window,P_", [(28, 4, 128, 64, None, 7), (28, 4, 128, 64, None, 2), (16, 1, 80, 32, 1000, 9), (14, 2, 64, 64, None, 8), (12, 2, 128, 64, None, 3),
                                                  (12, 2, 128, 64, None, 17), (14, 2, 64, 64, None, 1)])
def test_decode_attention_fused_of_many_sums(dtype, short, H, KV, hd, ps, window, P_):
    lens = [0, 1, 17, 31, 32, 33, 64, 95, 96, 126] if short else [0, 1, ps - 1, ps, 130, 700, 2049, 63, 64]
    ops = ops_for(dtype)
    splits = ops._decode_splits(len(lens), KV, max(-(-(c + 2) // ps) for c in lens), ps, window, ops._attention_lib(hd)[4], hd)
    assert (splits == 1) == short, f"{splits} splits: the sizes are those of the other form"
    _fused_decode_attention(dtype, H, KV, hd, ps, window, P_, lens)


def _fused_decode_attention(dtype, H, KV, hd, ps, window, P_, lens):
    ops, emu = ops_for(dtype), EmulatedOps(dtype)
    S = len(lens)
    gen = torch.Generator().manual_seed(600 + hd)
    n_pages = sum(-(-(c + 2) // ps) for c in lens) + 2
    order = torch.randperm(n_pages, generator=gen).tolist()
    kp, vp = rnd((n_pages, KV, ps, hd), dtype, 601), rnd((n_pages, KV, hd, ps), dtype, 602)
    width = max(-(-(c + 2) // ps) for c in lens)
    table = torch.full((S, width), -1, dtype=torch.int32)
    for i, c in enumerate(lens):
        for p in range(-(-(c + 2) // ps)):
            table[i, p] = order.pop()
    stride = (H + 2 * KV) * hd
    bias = rnd((stride,), torch.float32, 603)
    j = torch.arange(hd // 2, dtype=torch.float32)
    inv = 1.0 / torch.pow(torch.tensor(1e4), 2.0 * j / hd)
    kd, vd = kp.to(DEV), vp.to(DEV)
    for step in range(2):
        pos0 = torch.tensor([c + step for c in lens], dtype=torch.int32)
        slot_map = torch.tensor([int(table[i, (c + step) // ps]) * ps + (c + step) % ps for i, c in enumerate(lens)], dtype=torch.int32)
        qkv = rnd((S, stride), torch.float32, 604 + step)
        parts = torch.stack([qkv / P_ + (k - (P_ - 1) / 2) for k in range(P_)])  # P_ parts that sum to qkv
        ref = emu.decode_attention_fused(parts, bias, inv, slot_map, kp, vp, table, pos0, H, KV, hd, ps, window, hd ** -0.5)
        got = ops.decode_attention_fused(parts.to(DEV), bias.to(DEV), inv.to(DEV), slot_map.to(DEV), kd, vd, table.to(DEV),
                                         pos0.to(DEV), H, KV, hd, ps, window, hd ** -0.5)
        assert_close(got, ref, dtype, f"fused decode attention, step {step}")
        assert_close(kd, kp, dtype, "key pages")
        assert_close(vd, vp, dtype, "value pages")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,KV,hd,ps,window", [(14, 2, 64, 64, None), (4, 1, 128, 16, None), (6, 2, 64, 32, 4000)])
def test_attention_long_contexts(dtype, H, KV, hd, ps, window):
    """Contexts of nine and twenty thousand keys: a decoded row (many splits, merged in batches) and
    a portion of a prompt far into its request, with a key near the start (or at the window's
    edge) that towers over the rest, so that a range of keys that went missing would show."""
    ops, emu = ops_for(dtype), EmulatedOps(dtype)
    lens = [20011, 9000, 5]
    S = len(lens)
    gen = torch.Generator().manual_seed(700 + hd)
    n_pages = sum(-(-(c + 1) // ps) for c in lens) + 2
    order = torch.randperm(n_pages, generator=gen).tolist()
    kp, vp = rnd((n_pages, KV, ps, hd), dtype, 701), rnd((n_pages, KV, hd, ps), dtype, 702)
    width = max(-(-(c + 1) // ps) for c in lens)
    table = torch.full((S, width), -1, dtype=torch.int32)
    for i, c in enumerate(lens):
        for p in range(-(-(c + 1) // ps)):
            table[i, p] = order.pop()
    q = rnd((S, H * hd), dtype, 703)
    for i in (0, 1):
        far = 2 if not window else lens[i] - window + 1
        qv = q[i, (H - 1) * hd:].float()
        kp[int(table[i, far // ps]), KV - 1, far % ps, :] = (qv / qv.norm() * 8.0).to(dtype)
        q[i, (H - 1) * hd:] = (qv / qv.norm() * 8.0 * math.sqrt(hd) / 4).to(dtype)
    pos0 = torch.tensor(lens, dtype=torch.int32)
    ref = emu.decode_attention(q, kp, vp, table, pos0, H, KV, hd, ps, window, hd ** -0.5)
    got = ops.decode_attention(q.to(DEV), kp.to(DEV), vp.to(DEV), table.to(DEV), pos0.to(DEV), H, KV, hd, ps, window, hd ** -0.5)
    assert_close(got, ref, dtype, "decode attention over long contexts")
    # the last 150 positions of the 9,000-key request as one portion
    n, c = 150, lens[1] + 1 - 150
    g = H // KV
    qq = rnd((n, H * hd), dtype, 704)
    qq[n - 1] = q[1]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    emu.rows_per_block = ops.attention_rows_per_block(hd)
    args = (i32([0]), i32([n]), i32([c]), i32([(0, r0) for r0 in range(0, n * g, emu.rows_per_block)]).view(-1, 2))
    tab = table[1:2].contiguous()
    ref2 = emu.paged_attention(qq, kp, vp, tab, *args, H, KV, hd, ps, window, hd ** -0.5)
    got2 = ops.paged_attention(qq.to(DEV), kp.to(DEV), vp.to(DEV), tab.to(DEV), *[a.to(DEV) for a in args], H, KV, hd, ps,
                               window, hd ** -0.5)
    assert_close(got2, ref2, dtype, "a portion far into a long request")
    assert_close(got2[n - 1:].float().cpu(), got[1:2].float().cpu(), dtype, "its last row against the decode kernel")


@pytest.mark.parametrize("H,KV,hd,ps,T", [(4, 4, 32, 16, 50), (6, 2, 64, 32, 131), (3, 1, 48, 16, 70)])
def test_attention_equals_library_attention_without_rotation_or_paging(H, KV, hd, ps, T):
    """One request, its whole prompt in one step, pages in order: the kernel is plain causal attention,
    ``torch.nn.functional.scaled_dot_product_attention`` with the key/value heads repeated for their
    groups (head h reads key/value head h // g).  Then the last row again through the decode kernel."""
    import torch.nn.functional as F
    dtype, g = torch.float32, H // KV
    ops = ops_for(dtype)
    q, k, v = rnd((T, H, hd), dtype, 1), rnd((T, KV, hd), dtype, 2), rnd((T, KV, hd), dtype, 3)
    want = F.scaled_dot_product_attention(q.transpose(0, 1)[None].double(),
                                          k.transpose(0, 1).repeat_interleave(g, 0)[None].double(),
                                          v.transpose(0, 1).repeat_interleave(g, 0)[None].double(), is_causal=True)
    want = want[0].transpose(0, 1).reshape(T, H * hd).float()
    n_pages = -(-T // ps)
    kp, vp = torch.zeros(n_pages, KV, ps, hd), torch.zeros(n_pages, KV, hd, ps)
    for t in range(T):
        kp[t // ps, :, t % ps, :] = k[t]
        vp[t // ps, :, :, t % ps] = v[t]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table = i32(list(range(n_pages))).view(1, -1)
    work = i32([(0, r0) for r0 in range(0, T * g, ops.attention_rows_per_block(hd))]).view(-1, 2)
    got = ops.paged_attention(q.reshape(T, H * hd).to(DEV), kp.to(DEV), vp.to(DEV), table, i32([0]), i32([T]), i32([0]), work,
                              H, KV, hd, ps, None, hd ** -0.5)
    assert_close(got, want, dtype, "kernel against library attention")
    last = ops.decode_attention(q[T - 1:].reshape(1, H * hd).to(DEV), kp.to(DEV), vp.to(DEV), table, i32([T - 1]), H, KV, hd, ps,
                                None, hd ** -0.5)
    assert_close(last, want[T - 1:], dtype, "decode kernel against library attention")


@pytest.mark.parametrize("dtype", DTYPES)
def test_refusals(dtype):
    from machserve_amd.kernels import KernelError
    ops = ops_for(dtype)
    a, w = torch.zeros(4, 12, dtype=dtype, device=DEV), torch.zeros(16, 12, dtype=dtype, device=DEV)
    with pytest.raises(KernelError, match="multiple of 8"):
        ops.linear(a, w)
    with pytest.raises(Exception, match="multiple of 16"):
        ops.attention_rows_per_block(40)
    with pytest.raises(KernelError, match="GPU tensor"):
        ops.linear(a.cpu(), w)


def test_sampler_matches_cpu_mirror():
    """Peaked logits as in crates/mach-model/src/sampling.rs:1711-1752: the boundary tiers and
    the draw land far from any edge, so the orders of summation cannot change the outcome."""
    ops = ops_for(torch.float32)
    V, n = 2048, 12
    logits = torch.zeros(n, V)
    for s in range(n):
        logits[s] = 0.5 - 1.2 * torch.arange(V) * 0.25
        logits[s, ::37] += 0.05
        logits[s] = logits[s].roll(s * 97)
    temps = torch.tensor([[0.8, 1.0, 1.2, 0.0][i % 4] for i in range(n)])
    ks = torch.tensor([[0, 0, 40, 10][i % 4] for i in range(n)], dtype=torch.int32)
    ps_ = torch.tensor([[0.95, 1.0, 0.9, 0.8][i % 4] for i in range(n)])
    seeds = torch.tensor([7000 + i for i in range(n)], dtype=torch.int64)
    state = seeds.clone().to(DEV)
    for rep in range(3):
        got, _ = ops.sample(logits.to(DEV), temps.to(DEV), ks.to(DEV), ps_.to(DEV), state, any_greedy=rep != 1)
        for i in range(n):
            st = int(seeds[i]) + rep * P.RNG_GOLDEN
            want, new = P.sample(logits[i].numpy(), float(temps[i]), int(ks[i]), float(ps_[i]), st & P.MASK64)
            assert int(got[i]) == want, f"row {i} rep {rep}"
    want_state = [(int(s) + 3 * P.RNG_GOLDEN) & P.MASK64 for s in seeds]
    assert [int(v) & P.MASK64 for v in state.cpu().tolist()] == want_state


def test_sampler_draw_at_the_top_of_the_mass_falls_back_to_the_first_allowed_token():
    """A draw of u = 1 - 2^-24 (state 4375518: the finalizer's top 24 bits are all ones) on a row whose
    last segment is 64 tokens of probability 2^-26 behind a mass of one: each of them is lost when added
    to the running sum, so no walk passes the target, and the rule for that case decides: the first
    allowed token, then the maximum (crates/mach-model/src/sampling.rs:385-400).  In the second row the
    first allowed token is not the maximum: the kernel's rule gives token 0 where the reference's CPU
    mirror, which falls back to the maximum (sampling.rs:1270-1273), would give token 5."""
    ops = ops_for(torch.float32)
    assert P.next_uniform(4375518)[0] == 1.0 - 2.0 ** -24
    V = 1024 * 64
    tiny = -26.0 * 0.6931471805599453
    logits = torch.full((2, V), -200.0)
    logits[:, -64:] = tiny
    logits[0, 0] = 0.0                    # the maximum is also the first allowed token
    logits[1, 0], logits[1, 5] = tiny, 0.0
    state = torch.tensor([4375518, 4375518], dtype=torch.int64, device=DEV)
    got, _ = ops.sample(logits.to(DEV), torch.ones(2, device=DEV), torch.zeros(2, dtype=torch.int32, device=DEV),
                        torch.ones(2, device=DEV), state, any_greedy=False)
    assert got.cpu().tolist() == [0, 0]
    assert P.sample(logits[0].numpy(), 1.0, 0, 1.0, 4375518)[0] == 0     # the mirror agrees where the two rules do
    # a draw far from the top of the same rows walks as usual
    state = torch.tensor([5, 5], dtype=torch.int64, device=DEV)
    got, _ = ops.sample(logits.to(DEV), torch.ones(2, device=DEV), torch.zeros(2, dtype=torch.int32, device=DEV),
                        torch.ones(2, device=DEV), state, any_greedy=False)
    assert got.cpu().tolist() == [0, 5]


def test_sampler_greedy_ties_and_spread():
    ops = ops_for(torch.float32)
    V = 1000
    logits = torch.zeros(3, V)
    logits[0, [5, 700, 999]] = 2.0           # ties: the smallest index wins
    logits[1, 999] = 1.0
    logits[2] = torch.randn(V, generator=torch.Generator().manual_seed(1))
    z = torch.zeros(3)
    tok, lp = ops.sample(logits.to(DEV), z.to(DEV), torch.zeros(3, dtype=torch.int32, device=DEV), torch.ones(3).to(DEV),
                         torch.zeros(3, dtype=torch.int64, device=DEV))
    assert tok.cpu().tolist() == [5, 999, int(logits[2].argmax())]
    tok, lp = ops.sample(logits.to(DEV), z.to(DEV), torch.zeros(3, dtype=torch.int32, device=DEV), torch.ones(3).to(DEV),
                         torch.zeros(3, dtype=torch.int64, device=DEV), any_greedy=False)  # the one-block scan agrees
    assert tok.cpu().tolist() == [5, 999, int(logits[2].argmax())]
    big = torch.randn(5, 151936, generator=torch.Generator().manual_seed(2))
    big[3, [77, 150000]] = 9.0
    tok, _ = ops.sample(big.to(DEV), torch.zeros(5).to(DEV), torch.zeros(5, dtype=torch.int32, device=DEV), torch.ones(5).to(DEV),
                        torch.zeros(5, dtype=torch.int64, device=DEV))
    assert tok.cpu().tolist() == [int(big[i].argmax()) if i != 3 else 77 for i in range(5)]
    # the maximum at the borders of the chunks that the first stage cuts a row into, with rows that are 16-byte aligned
    # (a thread reads four entries at a time) and rows that are not
    for V2 in (1000, 1001, 777, 4096, 6002):
        chunk = -(-(-(-V2 // 64)) // 4) * 4
        places = sorted({0, 1, 3, 4, chunk - 1, chunk, chunk + 1, 2 * chunk - 1, 5 * chunk, V2 - 5, V2 - 4, V2 - 1} & set(range(V2)))
        rows = torch.randn(len(places), V2, generator=torch.Generator().manual_seed(V2))
        for i, at in enumerate(places):
            rows[i, at] = 30.0
            if at + 2 < V2:
                rows[i, at + 2] = 30.0           # a tie further on loses
        n = len(places)
        tok, _ = ops.sample(rows.to(DEV), torch.zeros(n).to(DEV), torch.zeros(n, dtype=torch.int32, device=DEV), torch.ones(n).to(DEV),
                            torch.zeros(n, dtype=torch.int64, device=DEV))
        assert tok.cpu().tolist() == places, f"vocabulary of {V2}"
    # a flat distribution is covered by different seeds
    flat = torch.zeros(64, V)
    st = torch.arange(1, 65, dtype=torch.int64).to(DEV)
    tok, _ = ops.sample(flat.to(DEV), torch.ones(64).to(DEV), torch.zeros(64, dtype=torch.int32, device=DEV),
                        torch.ones(64).to(DEV), st)
    assert len(set(tok.cpu().tolist())) > 40


def test_top_logprobs():
    """Ranked by probability, ties to the smaller id, logprob = log softmax at the row's temperature
    (crates/mach-model/src/sampling.rs:405-410)."""
    ops = ops_for(torch.float32)
    V = 5000
    logits = torch.randn(4, V, generator=torch.Generator().manual_seed(3)) * 3
    logits[1, [10, 4000, 77]] = 20.0     # a three-way tie at the top: ids ascending
    logits[2] = 0.0                      # all equal: the first ids
    inv_t = torch.tensor([1.0, 0.5, 2.0, 1.25])
    tok, lp = ops.top_logprobs(logits.to(DEV), inv_t.to(DEV), 20)
    tok, lp = tok.cpu(), lp.cpu()
    assert tok.shape == (4, 20)
    assert tok[1, :3].tolist() == [10, 77, 4000] and tok[2].tolist() == list(range(20))
    ref = torch.log_softmax(logits.double() * inv_t.double()[:, None], -1)
    for r in range(4):
        order = sorted(range(V), key=lambda i: (-logits[r, i].item(), i))[:20]
        assert tok[r].tolist() == order
        assert (lp[r].double() - ref[r, order]).abs().max() < 1e-4
    tok3, _ = ops.top_logprobs(logits.to(DEV), inv_t.to(DEV), 3)
    assert tok3.shape == (4, 3) and torch.equal(tok3.cpu(), tok[:, :3])


def test_feed_tokens():
    """The rows of a step whose input the step before it sampled take it on the device: listed rows only, entries of
    row -1 (the list is filled up to a fixed length) and anything outside either buffer change nothing."""
    ops = ops_for(torch.float32)
    tokens = torch.arange(100, 120, dtype=torch.int32, device=DEV)
    sampled = torch.tensor([7, 8, 9, 10, 11], dtype=torch.int32, device=DEV)
    rows = torch.tensor([3, 0, 19, -1, -1, 25, 4, -1], dtype=torch.int32, device=DEV)
    src = torch.tensor([4, 0, 2, 1, 0, 1, 9, 0], dtype=torch.int32, device=DEV)
    ops.feed_tokens(tokens, sampled, rows, src)
    want = list(range(100, 120))
    want[3], want[0], want[19] = 11, 7, 9       # row 25 is beyond the tokens, sample 9 beyond the samples
    assert tokens.cpu().tolist() == want


def test_logit_edit():
    ops = ops_for(torch.float32)
    x = torch.zeros(2, 10, device=DEV)
    ops.logit_edit(x, torch.tensor([0, 1, 1], dtype=torch.int32, device=DEV),
                   torch.tensor([3, 0, 9], dtype=torch.int32, device=DEV), torch.tensor([1.5, -2.0, 4.0], device=DEV))
    ref = torch.zeros(2, 10)
    ref[0, 3], ref[1, 0], ref[1, 9] = 1.5, -2.0, 4.0
    assert torch.equal(x.cpu(), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,H,KV,hd,K,ps", [(260, 3, 1, 64, 136, 16), (300, 14, 2, 64, 896, 64), (530, 4, 4, 64, 264, 32),
                                            (2048, 14, 2, 64, 896, 64), (1100, 12, 3, 64, 200, 64), (3000, 14, 2, 64, 896, 64)])
def test_qkv_product_that_rotates_and_writes_the_cache(dtype, M, H, KV, hd, K, ps):
    """The q/k/v projection of a step of many rows with bias, rotation and cache write in its epilogue: the same queries
    and the same pages as the plain product (32-bit sums) followed by the rotation kernel, and as the plain formulas
    (crates/mach-model/src/batched.rs:3566-3679); rows with a negative slot leave the pages alone; positions that are
    not the rows' indices."""
    ops = ops_for(dtype)
    assert ops.qkv_rope_takes(M, H, KV, hd, K) and not ops.qkv_rope_takes(256, H, KV, hd, K)
    assert not ops.qkv_rope_takes(M, H, KV, 80, K) and not ops.qkv_rope_takes(M, H, KV, 128, K)   # other heads: the two kernels
    N = (H + 2 * KV) * hd
    a, w, bias = rnd((M, K), dtype, 1), rnd((N, K), dtype, 2, K ** -0.5), rnd((N,), torch.float32, 3)
    gen = torch.Generator().manual_seed(4)
    positions = torch.randint(0, 5000, (M,), generator=gen, dtype=torch.int32)
    pages = -(-M // ps) + 2
    slots = torch.randperm(pages * ps, generator=gen)[:M].to(torch.int32)
    slots[5] = -1                                    # a row that writes nothing
    inv_freq = (1.0 / (10000.0 ** (torch.arange(hd // 2, dtype=torch.float32) * 2 / hd)))
    dev = lambda t: t.to(DEV)
    kp0, vp0 = rnd((pages, KV, ps, hd), dtype, 5), rnd((pages, KV, hd, ps), dtype, 6)
    # the two kernels it replaces
    kp1, vp1 = dev(kp0).clone(), dev(vp0).clone()
    sums = ops.linear(dev(a), dev(w), None, out_f32=True)
    q1 = ops.rope_kv_write(sums, dev(bias), dev(positions), dev(inv_freq), dev(slots), kp1, vp1, H, KV, hd, ps)
    # the one kernel
    kp2, vp2 = dev(kp0).clone(), dev(vp0).clone()
    table = ops.rope_table(dev(positions), dev(inv_freq))
    ang = positions.double()[:, None] * inv_freq.double()[None, :]
    assert (table[..., 0].cpu().double() - torch.cos(ang)).abs().max() < 1e-3 and (table[..., 1].cpu().double() - torch.sin(ang)).abs().max() < 1e-3
    q2 = ops.linear_qkv_rope(dev(a), dev(w), dev(bias), table, dev(slots), kp2, vp2, H, KV, hd, ps)
    assert_close(q2, q1.double(), dtype, "queries against the two kernels")
    assert_close(kp2, kp1.double(), dtype, "key pages against the two kernels")
    assert_close(vp2, vp1.double(), dtype, "value pages against the two kernels")
    # the plain formulas
    x = P.linear(a.double(), w.double(), bias.double())
    qr = P.rope(x[:, :H * hd].view(M, H, hd).float(), positions.long(), 10000.0).reshape(M, H * hd)
    assert_close(q2, qr.double(), dtype, "queries against the plain rotation")
    kr = P.rope(x[:, H * hd:(H + KV) * hd].view(M, KV, hd).float(), positions.long(), 10000.0)
    t = 17
    page, off = int(slots[t]) // ps, int(slots[t]) % ps
    assert_close(kp2[page, :, off, :], kr[t].double(), dtype, "a key in its page")
    assert_close(vp2[page, :, :, off], x[t, (H + KV) * hd:].view(KV, hd), dtype, "a value in its page")
    # what no row writes stays as it was (the row with the negative slot, and the slots nobody has)
    written = torch.zeros(pages * ps, dtype=torch.bool)
    written[slots[slots >= 0].long()] = True
    keep = (~written).view(pages, ps)
    assert torch.equal(kp2.cpu().permute(0, 2, 1, 3)[keep], kp0.permute(0, 2, 1, 3)[keep])
    assert torch.equal(vp2.cpu().permute(0, 3, 1, 2)[keep], vp0.permute(0, 3, 1, 2)[keep])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(16, 256), (1000, 320), (200, 4160), (5632, 1024), (40, 16384), (20000, 576)])
def test_products_whose_waves_share_out_k(dtype, M, N, K):
    """Few rows over whole K steps: one step a wave, waves with unequal numbers of steps, outputs that end inside a tile, one to many blocks a
    CU, with and without slices of K; every epilogue.  The sums are 32-bit: what differs from 64 bits is the order (1e-6 of the terms' size)."""
    from machserve_amd.kernels import interleave_gate_up
    ops = ops_for(dtype)
    a, w, bias = rnd((M, K), dtype, 71), rnd((N, K), dtype, 72, K ** -0.5), rnd((N,), torch.float32, 73)
    ref = P.linear(a.double(), w.double())
    ad, wd = a.to(DEV), w.to(DEV)
    if M <= 16:
        assert ops._few(M, N, K, True) and ops._few(M, N, K, False)
    parts = ops.linear_split(ad, wd)
    assert_close(parts.sum(0), ref, dtype, "slices")
    assert_close(ops.linear(ad, wd, None, out_f32=True), ref, dtype, "whole")
    assert_close(ops.linear(ad, wd, bias.to(DEV)), ref + bias.double(), dtype, "with a bias, in the element type")
    assert_close(ops.linear_act(ad, wd, "relu2"), torch.relu(ref) ** 2, dtype, "activation")
    x0 = rnd((M, N), torch.float32, 74)
    x = x0.to(DEV)
    pend = ops.linear_residual(ad, wd, x)
    assert_close(x.cpu() - x0 if pend is None else pend.sum(0), ref, dtype, "into the stream")
    g, u = rnd((N // 2 + 3, K), dtype, 75, 2 * K ** -0.5), rnd((N // 2 + 3, K), dtype, 76, K ** -0.5)
    gated = P.silu(P.linear(a.double(), g.double())) * P.linear(a.double(), u.double())
    gu = interleave_gate_up(g, u).to(DEV)
    assert_close(ops.linear_swiglu(ad, gu, N // 2 + 3), gated, dtype, "gated")
    if M <= 16:
        assert parts.shape[0] == ops.linear_split(ad[:1].contiguous(), wd).shape[0], "as many slices as for one row"
    if M <= 16 and ops._few(M, N, K, True) and parts.shape[0] == ops.linear_split(ad[:1].contiguous(), wd).shape[0]:
        assert torch.equal(parts[:, :1], ops.linear_split(ad[:1].contiguous(), wd)), "a row's sums do not depend on the other rows"
    if dtype == torch.bfloat16 and ops._plan("ms_prenorm_parts", M, N, K):
        xd, nw = x0.to(DEV).clone(), 1 + rnd((N,), torch.float32, 77, 0.1)
        hn, ss = ops.linear_residual_prenorm(ad, wd, xd, nw.to(DEV))
        assert_close(xd, x0.double() + ref, dtype, "stream")
        assert_close(hn, xd.cpu().double() * nw.double(), dtype, "stream times the norm's weight")
        assert_close(ss.sum(0), (xd.cpu().double() ** 2).sum(1), torch.float32, "sums of squares")
    if dtype == torch.bfloat16 and ops._plan("ms_swiglu_scaled_takes", M, N // 2 + 3, K):
        share = rnd((5, M), torch.float32, 78).abs() * K
        f = 1.0 / torch.sqrt(share.double().sum(0) / K + 1e-5)[:, None]
        scaled = P.silu(P.linear(a.double(), g.double()) * f) * (P.linear(a.double(), u.double()) * f)
        assert_close(ops.linear_swiglu_scaled(ad, share.to(DEV), 1e-5, gu, N // 2 + 3), scaled, dtype, "gated with row factors")


@pytest.mark.parametrize("M", [13, 16])
@pytest.mark.parametrize("N,K", [(4240, 1024), (9456, 256), (4104, 320)])
def test_sums_of_squares_of_a_last_block_that_is_part_full(M, N, K):
    """Widths whose blocks take two or four tiles of 16 columns and whose last block has fewer: nothing is written behind the parts that the plan
    states, and the parts add up to the rows' squares."""
    ops = ops_for(torch.bfloat16)
    a, w = rnd((M, K), torch.bfloat16, 81).to(DEV), rnd((N, K), torch.bfloat16, 82, K ** -0.5).to(DEV)
    x0, nw = rnd((M, N), torch.float32, 83), (1 + rnd((N,), torch.float32, 84, 0.1)).to(DEV)
    parts = ops._plan("ms_prenorm_parts", M, N, K)
    assert parts == -(-N // 16)
    x, hn, room = x0.to(DEV), torch.empty((M, N), dtype=torch.bfloat16, device=DEV), torch.full(((parts + 4) * M,), -7.0, device=DEV)
    from machserve_amd.kernels.ops import _c_int, _ptr
    ops._check(ops._core, ops._core.ms_linear_residual_prenorm(_ptr(a), _ptr(w), _ptr(x), _ptr(nw), _ptr(hn), _ptr(room), _c_int(M), _c_int(N),
                                                               _c_int(K), ops._stream()))
    assert bool((room[parts * M:] == -7.0).all())
    assert_close(x, x0.double() + P.linear(a.cpu().double(), w.cpu().double()), torch.bfloat16, "stream")
    assert_close(room[:parts * M].view(parts, M).sum(0), (x.cpu().double() ** 2).sum(1), torch.float32, "sums of squares")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 896, 896), (3, 1000, 320), (6, 448, 1024), (4, 72, 2048)])
def test_few_rows_whose_operands_begin_at_any_multiple_of_eight_bytes(dtype, M, N, K):
    """Operands that are views into a buffer: products that no tile is the choice for are taken as they lie, whole K steps or not."""
    from machserve_amd.kernels import interleave_gate_up
    ops = ops_for(dtype)
    if ops._tiled(M, N, K):
        pytest.skip("a tile is the choice for this one, whose operands are aligned")

    def off(t):  # the same numbers eight bytes behind a multiple of sixteen
        room = torch.empty(t.numel() + 12, dtype=t.dtype, device=DEV)
        at = 4 if room.data_ptr() % 16 == 0 else 0
        room[at:at + t.numel()] = t.flatten().to(DEV)
        return room[at:at + t.numel()].view(t.shape)

    a, w, x0, nw = rnd((M, K), dtype, 91), rnd((N, K), dtype, 92, K ** -0.5), rnd((M, N), torch.float32, 93), 1 + rnd((N,), torch.float32, 94, 0.1)
    g, u = rnd((N, K), dtype, 95, K ** -0.5), rnd((N, K), dtype, 96, K ** -0.5)
    ref, ad, wd, gu = P.linear(a.double(), w.double()), off(a), off(w), off(interleave_gate_up(g, u))
    assert ad.data_ptr() % 16 == 8 and wd.data_ptr() % 16 == 8 and ad.is_contiguous()
    assert_close(ops.linear_split(ad, wd).sum(0), ref, dtype, "slices")
    assert_close(ops.linear(ad, wd, None, out_f32=True), ref, dtype, "whole")
    assert_close(ops.linear_act(ad, wd, "relu2"), torch.relu(ref) ** 2, dtype, "activation")
    x = x0.to(DEV)
    pend = ops.linear_residual(ad, wd, x)
    assert_close(x.cpu() - x0 if pend is None else pend.sum(0), ref, dtype, "into the stream")
    pg, pu = P.linear(a.double(), g.double()), P.linear(a.double(), u.double())
    assert_close(ops.linear_swiglu(ad, gu, N), P.silu(pg) * pu, dtype, "gated")
    if ops._plan("ms_skinny_prenorm_parts", M, N, K):
        xd = x0.to(DEV)
        hn, ss = ops.linear_residual_prenorm(ad, wd, xd, nw.to(DEV))
        assert_close(xd, x0.double() + ref, dtype, "stream")
        assert_close(ss.sum(0), (xd.cpu().double() ** 2).sum(1), torch.float32, "sums of squares")
    if ops._plan("ms_swiglu_scaled_skinny_takes", M, N, K):
        share = rnd((5, M), torch.float32, 97).abs() * K
        f = 1.0 / torch.sqrt(share.double().sum(0) / K + 1e-5)[:, None]
        assert_close(ops.linear_swiglu_scaled(ad, share.to(DEV), 1e-5, gu, N), P.silu(pg * f) * (pu * f), dtype, "gated with row factors")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,d", [(1, 8), (3, 896), (2, 1024), (5, 1032), (4, 2048), (1, 2052), (7, 4096), (2, 4100), (3, 6)])
def test_embedding_rows_in_both_types(dtype, T, d):
    """One, two and four groups of 1,024 columns, widths behind them and widths that are no whole fours: rows in 32 bits and in the element type."""
    ops = ops_for(dtype)
    table, tokens = rnd((50, d), dtype, 101).to(DEV), torch.tensor([49, 0, 7, 7, 31, 2, 48][:T], dtype=torch.int32, device=DEV)
    for scale in (1.0, 3.0):
        ref = table[tokens.long()].float() * scale
        x, rounded = ops.embed_rounded(tokens, table, scale)
        assert torch.equal(x, ref) and torch.equal(rounded, ref.to(dtype))
        assert torch.equal(ops.embed(tokens, table, scale), ref)


def test_zeroing_a_place_of_several_arrays():
    """Arrays of unequal types and sizes, some no multiple of sixteen bytes: the place is zeros, its neighbours stay, a place that is not there is refused."""
    from machserve_amd.kernels import KernelError
    ops = ops_for(torch.bfloat16)
    arrays = [torch.ones((4, *s), dtype=t, device=DEV) for s, t in [((3,), torch.float32), ((16, 128, 128), torch.float32), ((1,), torch.int32), ((5, 7), torch.bfloat16), ((2048,), torch.float32)]]
    places = ops.places_of(arrays)
    for place in (2, 0, 3):
        ops.zero_places(places, place)
        for a in arrays:
            assert not bool(a[place].any()) and bool((a[1] == 1).all()) and bool((a[:place][[i not in (0, 2) for i in range(place)]] == 1).all())
    for place in (4, -1):
        with pytest.raises(KernelError):
            ops.zero_places(places, place)


@pytest.mark.parametrize("dtype", [torch.float64, torch.bfloat16])
def test_zeroing_a_slot_of_a_cache(dtype):
    """Whatever the cache's element type, one that has no kernels included: a slot's states in every layer are zeros, the others stay."""
    from machserve_amd.cache import CacheManager, DeviceCache
    from machserve_amd.parts.base import StateRequest
    cache = DeviceCache(CacheManager([StateRequest({"s": (3, 5), "c": (7,)}), StateRequest({"s": (16, 4)})], 16, 8, 2), dtype, torch.device(DEV))
    arrays = [t for layer in (0, 1) for t in cache.binding(layer).tensors.values()]
    for t in arrays:
        t.fill_(1)
    cache.zero_state(1)
    for t in arrays:
        assert not bool(t[1].any()) and bool((t[[0, 2]] == 1).all())


@pytest.mark.parametrize("d", [4, 896, 1024, 1028, 2048, 2052, 4096, 4100])
@pytest.mark.parametrize("na,nb", [(1, 1), (2, 1), (3, 2), (8, 8), (9, 1)])
def test_normed_branches_added_to_the_stream(d, na, nb):
    """One, two and four groups of 1,024 columns and widths behind them; up to two, up to eight and more sums: a branch, a branch with a bias, two branches weighed."""
    _normed_branches(3, d, na, nb)


@pytest.mark.parametrize("T,d,na,nb", [(3, 1024, 4, 4), (3, 2048, 4, 1), (3, 1028, 5, 3), (1024, 2048, 5, 1), (1025, 2048, 8, 5), (1025, 1028, 6, 1), (1025, 1024, 8, 8),
                                         (1024, 512, 4, 1), (1025, 512, 4, 2), (3, 512, 5, 1), (3, 516, 5, 5)])
def test_normed_branches_of_four_sums_and_of_many_rows(T, d, na, nb):
    """Up to four sums, and more than four of wide rows around four rows a CU; widths of which half of the threads have no columns."""
    _normed_branches(T, d, na, nb)


def _normed_branches(T, d, na, nb):
    ops, eps = ops_for(torch.bfloat16), 1e-5
    x0, pa, pb = rnd((T, d), torch.float32, 111), rnd((na, T, d), torch.float32, 112), rnd((nb, T, d), torch.float32, 113)
    w, bias = 1 + rnd((d,), torch.float32, 114, 0.2), rnd((d,), torch.float32, 115)
    norm = lambda y: y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps) * w.double()  # noqa: E731
    dev = lambda t: t.to(DEV)  # noqa: E731
    x = dev(x0)
    ops.norm_add(x, dev(pa), dev(w), eps)
    assert_close(x, x0.double() + norm(pa.double().sum(0)), torch.float32, "a branch")
    x = dev(x0)
    ops.norm_add_bias(x, dev(pa), dev(bias), dev(w), eps)
    assert_close(x, x0.double() + norm(pa.double().sum(0) + bias.double()), torch.float32, "a branch with a bias")
    x = dev(x0)
    ops.norm_add_weighted(x, dev(pa), 1.2, dev(pb), 0.7, dev(w), eps)
    assert_close(x, x0.double() + norm(1.2 * pa.double().sum(0) + 0.7 * pb.double().sum(0)), torch.float32, "two branches")
