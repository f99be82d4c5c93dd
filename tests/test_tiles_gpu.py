"""The tiles that products of more than 64 rows run in: every one at sizes that are no multiple of it, with one K step, two, three and
more (odd and even), in each epilogue; and a row's sums, which are the same whatever tile its batch runs in."""
import pytest
import torch

from gpu_util import DEV, assert_close

pytestmark = pytest.mark.gpu

# rows, columns, K, the tile of the plain product: 256x256, 256x192, 256x128, 128x128, 64x64, 64x64 with four buffers
SIZES = [(1537, 8200, 1024, 0), (1537, 8200, 1088, 0), (1000, 8200, 1024, 1), (1025, 8200, 1088, 1), (700, 6152, 1024, 2), (511, 8200, 1088, 2),
         (1000, 4104, 320, 3), (513, 8200, 384, 3), (193, 4104, 64, 4), (65, 2056, 64, 4), (1537, 130, 64, 4), (130, 8200, 192, 4),
         (65, 40, 64, 5), (193, 40, 192, 5), (127, 40, 128, 5)]


def rnd(shape, dtype, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


def ops_for(dtype):
    from machserve_amd.kernels import get_ops
    return get_ops(dtype, DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,tile", SIZES)
def test_products_in_every_tile(dtype, M, N, K, tile):
    from machserve_amd.kernels.ops import interleave_gate_up
    ops = ops_for(dtype)
    assert ops._plan("ms_tiled_tile", M, N, K, 1, 1) == tile, "the sizes are those of another tile"
    a, w, bias, x = rnd((M, K), dtype, 1), rnd((N, K), dtype, 2, K ** -0.5), rnd((N,), torch.float32, 3), rnd((M, N), torch.float32, 4)
    ref = a.float() @ w.float().T
    out = ops.linear(a, w, None, out_f32=True)
    assert_close(out, ref, torch.float32, "32-bit sums")
    assert_close(ops.linear(a, w, bias), ref + bias, dtype, "element type, with bias")
    assert_close(ops.linear_split(a, w).sum(0), ref, torch.float32, "sums in slices of K")
    assert_close(ops.linear_act(a, w, "relu2"), torch.relu(ref) ** 2, dtype, "activation in the epilogue")
    x1 = x.clone()
    pending = ops.linear_residual(a, w, x1)
    assert_close(x1 if pending is None else x1 + pending.sum(0), x + ref, torch.float32, "added to the stream")
    gate, up = w[:N // 2].contiguous(), w[N // 2:N // 2 * 2].contiguous()
    z, u = a.float() @ gate.float().T, a.float() @ up.float().T
    assert_close(ops.linear_swiglu(a, interleave_gate_up(gate, up), N // 2), z * torch.sigmoid(z) * u, dtype, "gated product")
    # the same rows in a batch of another size, another tile: the same sums bit for bit
    some = ops.linear(a[:65].contiguous(), w, None, out_f32=True)
    assert torch.equal(some, out[:65])


# Gated products in 256x320 tiles, a pair of gate and up tiles in every two waves: whole tiles, ragged at both edges, a single row in the last tile; K steps even and odd
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K", [(2048, 4800, 896), (1990, 4850, 960), (1985, 4850, 1024), (3001, 2811, 1024), (1793, 4864, 896)])
def test_gated_products_in_the_widest_tiles(dtype, act, M, I, K):
    from machserve_amd.kernels.ops import interleave_gate_up
    ops = ops_for(dtype)
    a, gate, up = rnd((M, K), dtype, 8), rnd((I, K), dtype, 9, 2 * K ** -0.5), rnd((I, K), dtype, 10, K ** -0.5)
    w = interleave_gate_up(gate, up)
    assert ops._plan("ms_gated_tile", M, w.shape[0], K) == 6, "the sizes are those of another tile"
    z, u = a.float() @ gate.float().T, a.float() @ up.float().T
    got = ops.linear_swiglu(a, w, I, act)
    assert_close(got, (torch.nn.functional.silu(z) if act == "silu" else torch.nn.functional.gelu(z, approximate="tanh")) * u, dtype, "gated product")
    assert torch.equal(ops.linear_swiglu(a[:300].contiguous(), w, I, act), got[:300]), "a row does not depend on its batch"


# 32-bit: tiles of 32x32 (gated products 32x64) and 64x64 with whole K steps, one to many of them, and a partial last step
@pytest.mark.parametrize("M,N,K", [(65, 40, 32), (97, 130, 64), (130, 200, 96), (501, 896, 160), (1025, 2056, 32), (1100, 2050, 352), (200, 136, 104)])
def test_32_bit_products_in_every_tile(M, N, K):
    from machserve_amd.kernels.ops import interleave_gate_up
    ops = ops_for(torch.float32)
    a, w, x = rnd((M, K), torch.float32, 5), rnd((N, K), torch.float32, 6, K ** -0.5), rnd((M, N), torch.float32, 7)
    ref = (a.double() @ w.double().T).float()
    out = ops.linear(a, w, None, out_f32=True)
    assert_close(out, ref, torch.float32, "sums")
    x1 = x.clone()
    assert ops.linear_residual(a, w, x1) is None
    assert_close(x1, x + ref, torch.float32, "added to the stream")
    gate, up = w[:N // 2].contiguous(), w[N // 2:N // 2 * 2].contiguous()
    z, u = a.double() @ gate.double().T, a.double() @ up.double().T
    assert_close(ops.linear_swiglu(a, interleave_gate_up(gate, up), N // 2), z * torch.sigmoid(z) * u, torch.float32, "gated product")
    assert torch.equal(ops.linear(a[:65].contiguous(), w, None, out_f32=True), out[:65]), "a row's sums do not depend on its batch"


# 32-bit products whose numbers are taken in parts of 16 bits: 64x64 and 128x128 tiles, one to many K steps, even and odd, ragged edges; K in slices, the last one short.
# The sums of many normal terms in 32 bits are off by sqrt(K) 2^-25 of their size, a slice's by less: within assert_close's 32-bit limit with room.
@pytest.mark.parametrize("M,N,K", [(193, 8200, 32), (200, 8202, 96), (321, 9000, 64), (330, 9008, 160), (65, 40, 4128), (130, 200, 4096), (900, 1030, 4160), (513, 896, 4864)])
def test_32_bit_products_in_parts(M, N, K):
    from machserve_amd.kernels.ops import interleave_gate_up
    ops = ops_for(torch.float32)
    a, w, x = rnd((M, K), torch.float32, 5), rnd((N, K), torch.float32, 6, K ** -0.5), rnd((M, N), torch.float32, 7)
    if N >= 4096:
        assert ops._plan("ms_parted", M, N, K, 1) == (2 if M > 300 else 1), "the sizes are those of another tile"
    else:
        slices = ops._plan("ms_residual_partials", M, N, K)
        assert slices > 1 and ops._plan("ms_parted", M, N, K, slices) > 0, "the sizes are those of an uncut product"
    ref = (a.double() @ w.double().T).float()
    def product():
        if N >= 4096:
            return ops.linear(a, w, None, out_f32=True)
        return ops.linear_residual(a, w, x).sum(0)

    out = product()
    assert_close(out, ref, torch.float32, "sums")
    if N >= 4096:
        x1 = x.clone()
        assert ops.linear_residual(a, w, x1) is None
        assert_close(x1, x + ref, torch.float32, "added to the stream")
    gate, up = w[:N // 2].contiguous(), w[N // 2:N // 2 * 2].contiguous()
    z, u = a.double() @ gate.double().T, a.double() @ up.double().T
    assert_close(ops.linear_swiglu(a, interleave_gate_up(gate, up), N // 2), z * torch.sigmoid(z) * u, torch.float32, "gated product")
    if M > 300 and N >= 4096:
        assert torch.equal(ops.linear(a[:193].contiguous(), w, None, out_f32=True), out[:193]), "a row's sums do not depend on the tile"
    # what is not finite, and a number whose first part is not, come out as in the 32-bit products
    a[3, 5], a[64, 7], w[9, 11] = float("inf"), float("nan"), float("-inf")
    w[:, 1] *= 1e-3  # (no sum of these is beyond 3.4e38 * 5e-3, in whatever order)
    a[:, 2] *= 1e-3
    a[20, 1], w[21, 2] = 3.4e38, 3.4e38
    got, ref = product(), a.double() @ w.double().T
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(got[~torch.isfinite(got)].nan_to_num(0.5), ref[~torch.isfinite(ref)].float().nan_to_num(0.5))
    fine = torch.isfinite(ref)
    err = (got.double() - ref).abs()[fine] / (a.abs().double().nan_to_num(0, 0, 0) @ w.abs().double().nan_to_num(0, 0, 0).T)[fine]
    assert float(err.max()) < 2e-6


# Below two tiles of 64x64 a CU, at two, behind them, towards three, at a few more: where the 32-bit instructions fill their rounds they stay.
@pytest.mark.parametrize("M,N,K,parts", [(160, 9728, 896, 0), (192, 9728, 896, 1), (512, 4096, 1024, 0), (400, 4864, 896, 1), (300, 9728, 896, 0), (400, 9728, 896, 1), (64, 9728, 896, 0)])
def test_which_32_bit_products_are_taken_in_parts(M, N, K, parts):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are those of 256 CUs")
    assert (ops_for(torch.float32)._plan("ms_parted", M, N, K, 1) > 0) == bool(parts)


# ... with nothing lost that the 32-bit products keep: a single product, small numbers of any scale, and rows beside ones that are not finite; both tiles, and K in slices
@pytest.mark.parametrize("M,N,K", [(193, 8200, 64), (330, 9008, 96), (65, 136, 4128), (513, 896, 4864)])
def test_32_bit_parts_lose_nothing(M, N, K):
    ops = ops_for(torch.float32)
    slices = ops._plan("ms_residual_partials", M, N, K)
    assert ops._plan("ms_parted", M, N, K, slices) > 0, "the sizes are those of the 32-bit instructions"
    x = torch.zeros((M, N), device=DEV)

    def product(a, w):
        return ops.linear(a, w, None, out_f32=True) if N >= 4096 else ops.linear_residual(a, w, x).sum(0)

    # one product a sum: rounded once, half a unit; what its parts add up to first is at most 2^-6 of it and rounded seven times
    a, w = torch.zeros((M, K), device=DEV), torch.zeros((N, K), device=DEV)
    a[:, 37], w[:, 37] = 1 + rnd((M,), torch.float32, 41).abs() % 1, 1 + rnd((N,), torch.float32, 42).abs() % 1
    ref = a.double() @ w.double().T
    err = float(((product(a, w).double() - ref).abs() / ref).max())
    assert err <= 2.0 ** -24 * (1 + 7 * 2.0 ** -6), f"a single product is off by {err:.3e}"

    # many: a slice's sum of n terms rounds n times at most, by a quarter of a unit on average, in no direction; sums of numbers of any size alike
    n, a, w = K // slices, rnd((M, K), torch.float32, 43), rnd((N, K), torch.float32, 44)
    for ea, ew in [(0, 0), (-118, 0), (-118, 118), (0, -122), (100, -122), (-60, -60), (-104, 4)]:
        sa, sw = (a.double() * 2.0 ** ea).float(), (w.double() * 2.0 ** ew).float()
        ref = sa.double() @ sw.double().T
        err = float((product(sa, sw).double() - ref).norm() / ref.norm())
        assert err <= n ** 0.5 * 2.0 ** -24, f"numbers of 2^{ea} and 2^{ew}: error {err:.3e}"

    # what stands in other rows of the block, and in other columns' weights, does not show
    want = product(a, w)
    odd, odd_w = a.clone(), w.clone()
    odd[3, 5], odd[20, 1], odd[64, 7], odd[M - 1] = float("inf"), 2.0 ** -120, float("nan"), odd[M - 1] * 2.0 ** -110
    odd_w[9, 11], odd_w[11] = float("-inf"), 0.0
    rows, cols = torch.ones(M, dtype=torch.bool, device=DEV), torch.ones(N, dtype=torch.bool, device=DEV)
    rows[[3, 20, 64, M - 1]], cols[[9, 11]] = False, False
    got = product(odd, odd_w)
    assert torch.equal(got[rows][:, cols], want[rows][:, cols])
    ref = odd.double() @ odd_w.double().T
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and bool((got[rows][:, 11] == 0).all())


# Around a norm, more than 64 rows: the product that prepares it in every tile, ragged at both edges, a last column of waves that has no columns (widths of 20 and 1,030); what
# the kernel leaves behind its last part stays untouched.
@pytest.mark.parametrize("M,N,K,tile", SIZES + [(1030, 1030, 512, None), (65, 20, 64, None), (200, 24, 128, None), (2048, 896, 896, None)])
def test_products_that_prepare_a_norm(M, N, K, tile):
    from machserve_amd.kernels.ops import _c_int, _ptr
    ops = ops_for(torch.bfloat16)
    a, w, x0 = rnd((M, K), torch.bfloat16, 21), rnd((N, K), torch.bfloat16, 22, K ** -0.5), rnd((M, N), torch.float32, 23)
    nw = 1 + rnd((N,), torch.float32, 24, 0.1)
    parts = ops._plan("ms_prenorm_parts", M, N, K)
    if ops._plan("ms_tiled_partials", M, N, K) > 1:
        assert parts == 0 and ops.linear_residual(a, w, x0.clone()) is not None
        return
    assert parts > 0
    want = x0.clone()
    assert ops.linear_residual(a, w, want) is None
    x, hn, room = x0.clone(), torch.empty((M, N), dtype=torch.bfloat16, device=DEV), torch.full(((parts + 4) * M,), -7.0, device=DEV)
    ops._check(ops._core, ops._core.ms_linear_residual_prenorm(_ptr(a), _ptr(w), _ptr(x), _ptr(nw), _ptr(hn), _ptr(room), _c_int(M), _c_int(N), _c_int(K), ops._stream()))
    assert torch.equal(x, want) and torch.equal(hn, (x * nw).bfloat16())
    assert bool((room[parts * M:] == -7.0).all())
    assert_close(room[:parts * M].view(parts, M).sum(0), (x.double() ** 2).sum(1), torch.float32, "sums of squares")


# ... and the gated product that applies the rows' factors, in every tile: one part and more than sixteen
@pytest.mark.parametrize("M,I,K,parts", [(2048, 4800, 896, 28), (1990, 4850, 960, 17), (1537, 4100, 1024, 1), (1000, 4100, 1024, 16), (700, 3076, 1024, 5), (1000, 2052, 320, 33),
                                         (193, 2052, 256, 4), (65, 1028, 256, 40), (130, 20, 320, 3), (512, 4864, 896, 28)])
def test_gated_products_with_row_factors_of_many_rows(M, I, K, parts):
    from machserve_amd.kernels.ops import interleave_gate_up
    ops = ops_for(torch.bfloat16)
    a, gate, up = rnd((M, K), torch.bfloat16, 31), rnd((I, K), torch.bfloat16, 32, 2 * K ** -0.5), rnd((I, K), torch.bfloat16, 33, K ** -0.5)
    w, share = interleave_gate_up(gate, up), rnd((parts, M), torch.float32, 34).abs() * K / parts
    f = 1.0 / torch.sqrt(share.double().sum(0) / K + 1e-5)[:, None]
    z, u = (a.double() @ gate.double().T) * f, (a.double() @ up.double().T) * f
    got = ops.linear_swiglu_scaled(a, share, 1e-5, w, I)
    assert_close(got, z * torch.sigmoid(z) * u, torch.bfloat16, "gated product with row factors")
    if M > 300:
        assert_close(ops.linear_swiglu_scaled(a[:200].contiguous(), share[:, :200].contiguous(), 1e-5, w, I), got[:200].double(), torch.bfloat16, "a row in another batch")


@pytest.mark.parametrize("M,width,I,pays", [(2048, 896, 4864, True), (2049, 896, 4864, False), (1024, 1536, 8960, True), (1500, 1536, 8960, False), (2048, 3584, 18944, False),
                                            (3001, 1024, 2816, True), (16, 896, 4864, True)])
def test_a_norm_is_prepared_where_the_gated_product_is_a_round(M, width, I, pays):
    """Around a round of the gated product's tiles; with either answer the norm between the products is the same."""
    from machserve_amd.kernels.ops import interleave_gate_up
    ops = ops_for(torch.bfloat16)
    assert ops.prenorm_swiglu_takes(M, width, width, 2 * I) == pays
    if M > 2049:
        return
    a, w, x = rnd((M, width), torch.bfloat16, 61), rnd((width, width), torch.bfloat16, 62, width ** -0.5), rnd((M, width), torch.float32, 63)
    gu, nw = interleave_gate_up(rnd((I, width), torch.bfloat16, 64, width ** -0.5), rnd((I, width), torch.bfloat16, 65, width ** -0.5)), 1 + rnd((width,), torch.float32, 66, 0.1)
    x1 = x.clone()
    assert ops._plan("ms_prenorm_parts", M, width, width) > 0
    want = ops.linear_swiglu(ops.rmsnorm(x1, nw, 1e-6, partials=ops.linear_residual(a, w, x1)), gu, I)
    assert_close(ops.linear_swiglu_scaled(*ops.linear_residual_prenorm(a, w, x, nw), 1e-6, gu, I), want.float(), torch.bfloat16, "gated product behind a norm")
