"""Products over the rows that chose an expert, against the same feed-forward over every expert in 64 bits: steps of one tile an expert
and of lists, at the edges of both; experts that no row or every row uses; planes that a row does not use."""
import pytest
import torch

from emulated_ops import EmulatedOps
from gpu_util import DEV, assert_close

pytestmark = pytest.mark.gpu

# rows, router outputs, of them experts, used a row, columns of an expert, columns of the expert for every row, width
SIZES = [(1, 8, 8, 2, 64, 0, 128), (4, 9, 8, 2, 128, 64, 192), (64, 5, 5, 3, 64, 128, 64), (65, 5, 5, 3, 64, 64, 64), (129, 8, 6, 2, 192, 0, 256),
         (300, 70, 68, 1, 64, 0, 128), (700, 4, 3, 2, 128, 64, 320), (1025, 2, 2, 2, 64, 64, 64),
         (3100, 4, 4, 2, 1472, 64, 832), (4300, 2, 2, 1, 1984, 1024, 832), (40, 130, 130, 12, 64, 64, 64),
         # products of few rows: whole and partial rounds of the waves' K steps, 16, 17, 32 and 33 rows, most of an expert's rows and hardly any
         (1, 8, 8, 2, 256, 256, 256), (16, 9, 8, 2, 320, 256, 448), (17, 5, 5, 3, 256, 320, 576), (32, 2, 2, 2, 704, 0, 320), (33, 8, 8, 2, 256, 256, 256),
         (30, 40, 40, 1, 256, 0, 256)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,outputs,E,top,ff,shared,width", SIZES)
@pytest.mark.parametrize("kind", ["gated", "gated, weighed at the input", "plain"])
def test_products_over_the_rows_that_chose_an_expert(dtype, T, outputs, E, top, ff, shared, width, kind):
    from machserve_amd.kernels import get_ops
    from machserve_amd.kernels.ops import interleave_gate_up
    ops, gated, inside = get_ops(dtype, DEV), kind != "plain", kind.endswith("input")
    g = torch.Generator().manual_seed(T * 31 + E)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    h = rnd(T, width).to(dtype)
    shared_gate = bool(shared) and outputs == E
    router = rnd(outputs + shared_gate, width) * 0.3
    if E > 2:
        router[1] = -1e3 * h[T // 2].float() / h[T // 2].float().norm()  # hardly any row, or none, chooses this one
    cols = [ff] * E + ([shared] if shared else [])
    gate, up = [(rnd(c, width) * width ** -0.5).to(dtype) for c in cols], [(rnd(c, width) * width ** -0.5).to(dtype) for c in cols]
    down = [(rnd(width, c) * c ** -0.5).to(dtype) for c in cols]
    w_up = torch.cat([interleave_gate_up(a, b) if gated else b for a, b in zip(gate, up)])
    w_down = torch.cat(down, dim=1)
    scoring = {"sigmoid": True} if inside else ({"softmax_all": True} if outputs > E else {})
    sums, gates = ops.routed_experts(h.to(DEV), router.to(DEV), None, top, w_up.to(DEV), w_down.to(DEV), E, ff, shared, "silu", gated=gated,
                                     weigh_input=inside, shared_gate=shared_gate, **scoring)
    assert sums.shape == (top + (shared > 0), T, width) and bool(torch.isfinite(sums).all())
    # the weights themselves: the stand-in's on the CPU (32-bit sums in another order).  Each of two logits is off by up to 2^-23 of the
    # largest (the planted one, some thousands), and a weight's slope over their difference is at most 1/4
    weights = EmulatedOps(torch.float32).route(h.float(), router, None, top, extra_gates=int(shared_gate), **scoring)
    off = (h.double() @ router.double().T).abs().max().item() * 2 ** -22 / 4 + 2.1e-5
    assert (gates.cpu() - weights).abs().max().item() <= off, "weights"
    w = gates.double().cpu()
    want = torch.zeros(T, width, dtype=torch.float64)
    silu = lambda z: z * torch.sigmoid(z)  # noqa: E731
    for e in range(len(cols)):
        we = (w[:, e] if e < E or shared_gate else torch.ones(T, dtype=torch.float64))[:, None]
        wi = we if inside and e < E else 1.0
        a, b = h.double() @ gate[e].double().T, h.double() @ up[e].double().T
        z = silu(wi * a) * b * we if gated else silu(b) * we
        want += z.to(dtype).double() @ down[e].double().T  # the activations are kept in the element type
    assert_close(sums.sum(0), want, dtype, kind)
    used = (w[:, :E] != 0).sum(1)
    for k in range(top):
        assert not bool(sums[k].cpu()[used <= k].any()), "a plane that a row does not use is zero"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [3, 200])
@pytest.mark.parametrize("spec", [dict(gated=True, scoring="sigmoid", weigh="input", shared=64, shared_gate=True), dict(router_bias=True, shared=128),
                                  dict(gated=True, scoring="softmax_all", correction=True, identity=2), dict(gated=True, shared=64)])
def test_the_part_gives_what_it_gives_over_every_expert(dtype, T, spec, monkeypatch):
    """The same part with the same tensors: over the rows that chose an expert, and over every expert."""
    from machserve_amd.config import RoutedMlpSpec
    from machserve_amd.kernels import get_ops
    from machserve_amd.parts import FEED_FORWARDS, Runtime
    from machserve_amd.parts.base import ResidualStream
    ops, spec = get_ops(dtype, DEV), dict(spec)
    width, E, top, ff, shared, bias = 128, 6, 2, 64, spec.pop("shared", 0), spec.pop("router_bias", False)
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, width, generator=g).to(dtype).to(DEV)
    x = torch.randn(T, width, generator=g).to(DEV)
    tensors, got = {}, []
    for takes in (True, False):
        monkeypatch.setattr(ops, "routed_experts_takes", lambda *a, takes=takes: takes)
        part = FEED_FORWARDS.build(RoutedMlpSpec("routed_mlp", width, E, top, ff, "silu", shared, bias, {}, **spec), Runtime(torch.device(DEV), dtype, ops))
        for d in part.tensor_decls():
            if d.name not in tensors:
                tensors[d.name] = (torch.randn(d.shape, generator=g) * 0.1).to(DEV, torch.float32 if d.role == "vector" else dtype)
        part.load(tensors)
        assert part.grouped == takes
        stream = ResidualStream(x.clone(), ops)
        part.forward(h, stream, None)
        got.append(stream.value())
    assert_close(got[0], got[1], dtype, str(spec))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [3, 200])
@pytest.mark.parametrize("block", ["postnorm", "sandwich"])
@pytest.mark.parametrize("top,shared", [(1, 0), (2, 64), (6, 64)])
def test_the_norm_behind_the_experts(dtype, T, block, top, shared, monkeypatch):
    """The feed-forward of a block whose norm stands behind it: the experts' planes (up to four, which that norm adds together with the
    next one, and more) against the operands of one product."""
    from machserve_amd.config import NormSpec, RoutedMlpSpec
    from machserve_amd.kernels import get_ops
    from machserve_amd.parts import FEED_FORWARDS, NORMS, Runtime
    from machserve_amd.parts.base import ResidualStream
    from machserve_amd.parts.block import PostNormBlock, SandwichBlock
    ops, width, E, ff = get_ops(dtype, DEV), 128, 7, 64
    g, rt = torch.Generator().manual_seed(T + top), Runtime(torch.device(DEV), dtype, ops)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, tensors, got = rnd(T, width).to(DEV), {}, []
    pre, post, after = (NORMS.build(NormSpec("rmsnorm", width, 1e-5, {}), rt) for _ in range(3))
    for norm in (pre, post, after):
        norm.load({"weight": (1 + 0.1 * rnd(width)).to(DEV)})
    for takes in (True, False):
        monkeypatch.setattr(ops, "routed_experts_takes", lambda *a, takes=takes: takes)
        part = FEED_FORWARDS.build(RoutedMlpSpec("routed_mlp", width, E, top, ff, "silu", shared, False, {}, gated=True), rt)
        for d in part.tensor_decls():
            if d.name not in tensors:
                tensors[d.name] = (rnd(*d.shape) * 0.1).to(DEV, torch.float32 if d.role == "vector" else dtype)
        part.load(tensors)
        assert part.grouped == takes
        kind = {"postnorm": PostNormBlock, "sandwich": SandwichBlock}[block]
        own, stream = kind.__new__(kind), ResidualStream(x.clone(), ops)
        own.rt = rt
        own._branch(*([part, post] if block == "postnorm" else [pre, part, post]), stream, None)
        got.append((after.forward(stream), stream.value()))
    assert_close(got[0][0], got[1][0], dtype, "the next norm's rows")
    assert_close(got[0][1], got[1][1], dtype, "the stream")


@pytest.mark.parametrize("T", [1, 2, 63, 64])
@pytest.mark.parametrize("shared", [0, 64])
def test_a_step_of_few_rows_sets_no_more_activations_aside_than_its_rows_could_fill(T, shared):
    """... for every expert, and for the one that every row uses: what the whole call holds at its most is that and what it returns."""
    from machserve_amd.kernels import get_ops
    ops, E, top, ff, width = get_ops(torch.bfloat16, DEV), 200, 2, 64, 64
    g = torch.Generator().manual_seed(T)
    h, router = torch.randn(T, width, generator=g).to(DEV, torch.bfloat16), torch.randn(E, width, generator=g).to(DEV)
    w_up, w_down = (torch.zeros(s, dtype=torch.bfloat16, device=DEV) for s in ((E * ff + shared, width), (width, E * ff + shared)))
    call = lambda: ops.routed_experts(h, router, None, top, w_up, w_down, E, ff, shared, "silu")  # noqa: E731
    call()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    call()
    torch.cuda.synchronize()
    rows = E * T + (T if shared else 0)
    # the activations; numbers and weights; the planes; a tensor is rounded up to 512 bytes
    assert torch.cuda.max_memory_allocated() - before <= rows * ff * 2 + 2 * T * E * 4 + (top + 1) * T * width * 4 + 4 * 512


# one row a block and four, a ragged last block; few outputs (one lane each), more than 64; columns that come in fours and that do not
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,top,d", [(1, 8, 2, 256), (5, 13, 13, 1030), (1023, 9, 2, 128), (1030, 64, 6, 192), (1025, 65, 5, 130), (3, 200, 64, 2048)])
@pytest.mark.parametrize("scoring", [{}, {"softmax_all": True}, {"sigmoid": True, "extra_gates": 3}])
def test_the_router_in_its_forms(dtype, T, E, top, d, scoring):
    from machserve_amd.kernels import get_ops
    g = torch.Generator().manual_seed(T + E)
    x, w = torch.randn(T, d, generator=g).to(dtype), torch.randn(E + scoring.get("extra_gates", 0), d, generator=g) * d ** -0.5
    w[E // 2] = w[0]  # two outputs that tie in every row: the first is chosen
    got = get_ops(dtype, DEV).route(x.to(DEV), w.to(DEV), None, top, **scoring).cpu()
    want = EmulatedOps(torch.float32).route(x.float(), w, None, top, **scoring)
    z = (x.double() @ w[:E].double().T).sort(1, descending=True).values
    # logits are 32-bit sums of d products: off by about sqrt(d) 2^-24 of their size; rows whose last chosen logit has a near equal may differ
    clear = torch.ones(T, dtype=torch.bool) if top == E else ((z[:, top - 1] - z[:, top]).abs() > 1e-5)
    assert clear.float().mean() > 0.5
    assert not bool(((got[:, E // 2] > 0) & (got[:, 0] == 0)).any()), "of equals the first"
    assert (got - want)[clear].abs().max().item() <= 1e-5


# at most four outputs, extra gates among them: a wave has one and not three; one row a block and four, columns in fours and not.  (With two outputs
# that tie, two thirds of the rows of three have no tie at the second place, and none matters where all are chosen.)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,top,d", [(1, 4, 2, 256), (1023, 3, 2, 130), (1030, 4, 4, 192), (1030, 2, 2, 1030)])
def test_the_router_of_few_outputs(dtype, T, E, top, d):
    from machserve_amd.kernels import get_ops
    test_the_router_in_its_forms(dtype, T, E, top, d, {"softmax_all": True})
    if E < 4:
        test_the_router_in_its_forms(dtype, T, E, top, d, {"sigmoid": True, "extra_gates": 4 - E})
    g = torch.Generator().manual_seed(E)
    x, w, bias = torch.randn(T, d, generator=g).to(dtype), torch.randn(5, d, generator=g) * d ** -0.5, torch.tensor([0.0] * E + [-1e4] * (5 - E))
    few, more = (get_ops(dtype, DEV).route(x.to(DEV), w[:n].contiguous().to(DEV), bias[:n].to(DEV), top) for n in (E, 5))
    assert torch.equal(few, more[:, :E]), "a logit does not depend on how many there are"


def test_the_router_refuses_numbers_and_sums_that_its_kernel_does_not_assume():
    from machserve_amd.kernels import KernelError, get_ops
    ops, new = get_ops(torch.bfloat16, DEV), lambda shape, dt: torch.zeros(shape, dtype=dt, device=DEV)  # noqa: E731
    T, d, E, top = 5, 64, 6, 3
    h, w = new((T, d), torch.bfloat16), new((E, d), torch.float32)
    plane, sums = new((T, E), torch.int32), new((top, T, d), torch.float32)
    for p, s in [(plane, None), (None, sums), (plane, sums[:top - 1]), (plane, sums[:, :T - 1].contiguous()), (plane, sums[..., :d // 2].contiguous()),
                 (plane, sums.transpose(1, 2).contiguous().transpose(1, 2)), (plane, sums.double()), (plane, sums.cpu()), (plane, sums[0]),
                 (plane[:T - 1], sums), (plane[0], sums), (plane.long(), sums), (plane.t().contiguous().t(), sums), (plane.cpu(), sums),
                 (new((T, E + 1), torch.int32), sums), (new((T, 0), torch.int32), sums)]:
        with pytest.raises(KernelError):
            ops.route(h, w, None, top, plane=p, sums=s)
    ops.route(h, w, None, top, plane=plane, sums=sums)
    assert plane.tolist() == [[0, 1, 2, -1, -1, -1]] * T  # equal logits: the lower index wins


@pytest.mark.parametrize("z0,z1", [(-60.0, -30.0), (-8.0, 8.0)])
def test_the_experts_silu_is_as_exact_as_32_bits_allow(z0, z1):
    """e^-z, the sum and the division are each right to about a unit of 32 bits, 2^-22 of the result together: it is rounded to another
    bfloat16 than the exact result where that lies so near to the middle of two of them (2^-8 apart or more), which is one number in 8,192."""
    from machserve_amd.kernels import get_ops
    n = 1 << 18
    z = torch.rand(1, n, generator=torch.Generator().manual_seed(11)) * (z1 - z0) + z0
    got = get_ops(torch.bfloat16, DEV).expert_act(z.to(DEV), torch.ones(1, 1, device=DEV), n, "silu").cpu()
    want = (z.double() / (1.0 + torch.exp(-z.double()))).to(torch.bfloat16)
    assert int((got != want).sum()) <= n // 8192
