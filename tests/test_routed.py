"""Routed experts under blocks, norms and collectors of every kind, at sizes where the products run over the rows that chose an expert: over
stand-ins that say so, the part gives what it gives over every expert, whoever takes its output."""
import pytest
import torch

from emulated_ops import EmulatedOps
from machserve_amd.config import NormSpec, RoutedMlpSpec
from machserve_amd.parts import FEED_FORWARDS, NORMS, Runtime
from machserve_amd.parts.base import ResidualStream
from machserve_amd.parts.block import PostNormBlock, SandwichBlock

WIDTH, E, TOP, FF, SHARED = 128, 5, 2, 64, 64


class GroupedOps(EmulatedOps):
    """Stand-ins whose experts run over the rows that chose them, as the kernels' do."""
    grouped_calls = 0

    def routed_experts_takes(self, width, ff, shared, top):
        return width % 64 == 0 and ff % 64 == 0 and shared % 64 == 0

    def routed_experts_runs(self, rows):
        return True

    def routed_experts(self, h, w_router, b_router, top, w_up, w_down, experts, ff, shared, activation, gated=False, weigh_input=False,
                       shared_gate=False, **scoring):
        self.grouped_calls += 1
        gates = self.route(h, w_router, b_router, top, extra_gates=int(shared_gate), **scoring)
        a = self.expert_act(h.float() @ w_up.float().t(), gates, ff, activation, experts=experts, gated=gated, weigh_input=weigh_input,
                            shared_gate=shared_gate, interleaved=True)
        sums = torch.zeros(top + (shared > 0), h.shape[0], h.shape[1])
        for t in range(h.shape[0]):
            for k, e in enumerate(torch.nonzero(gates[t, :experts]).flatten().tolist()):
                sums[k, t] = a[t, e * ff:(e + 1) * ff].float() @ w_down[:, e * ff:(e + 1) * ff].float().t()
        if shared:
            sums[top] = a[:, experts * ff:].float() @ w_down[:, experts * ff:].float().t()
        return sums, gates

    def expert_act(self, up, *args, interleaved=False, gated=False, **kw):
        if interleaved and gated:
            pairs = up.view(up.shape[0], -1, 2, 16)
            up = torch.cat([pairs[:, :, 0].reshape(up.shape[0], -1), pairs[:, :, 1].reshape(up.shape[0], -1)], 1)
        return super().expert_act(up, *args, gated=gated, **kw)


class _Products:
    """A collector that knows the operands of last products alone."""

    def add_linear(self, a, w, bias=None):
        self.y = a.float() @ w.float().t()


class _NormOfProducts:
    """A norm behind a branch with nothing but ``add_normed`` and ``add_normed_tensor``."""

    def __init__(self, norm):
        self.norm = norm
        self.add_normed, self.add_normed_tensor = norm.add_normed, norm.add_normed_tensor


def _part(ops, gated, g):
    rt = Runtime(torch.device("cpu"), torch.float32, ops)
    part = FEED_FORWARDS.build(RoutedMlpSpec("routed_mlp", WIDTH, E, TOP, FF, "silu", SHARED, False, {}, gated=gated), rt)
    part.load({d.name: torch.randn(d.shape, generator=g) * 0.1 for d in part.tensor_decls()})
    return part


def _both(gated):
    """The part with the same tensors over both kinds of stand-ins."""
    return [_part(ops, gated, torch.Generator().manual_seed(3)) for ops in (GroupedOps(), EmulatedOps())]


@pytest.mark.parametrize("gated", [False, True])
def test_a_collector_of_last_products_alone_is_served(gated):
    h, got = torch.randn(7, WIDTH, generator=torch.Generator().manual_seed(1)), []
    for part in _both(gated):
        out = _Products()
        part.forward(h, out, None)
        got.append(out.y)
    assert (got[0] - got[1]).abs().max() <= 1e-5 * got[1].abs().max()


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("block", [PostNormBlock, SandwichBlock])
@pytest.mark.parametrize("products_only", [False, True])
def test_the_norm_behind_a_branch(block, gated, products_only):
    """A norm that takes sums gets them; one that takes products alone gets the product over every expert."""
    x, got = torch.randn(7, WIDTH, generator=torch.Generator().manual_seed(2)), []
    for part in _both(gated):
        rt = part.rt
        pre, post = (NORMS.build(NormSpec("rmsnorm", WIDTH, 1e-5, {}), rt) for _ in range(2))
        for i, norm in enumerate((pre, post)):
            norm.load({"weight": torch.randn(WIDTH, generator=torch.Generator().manual_seed(i))})
        if products_only:
            post = _NormOfProducts(post)
        own, stream = block.__new__(block), ResidualStream(x.clone(), rt.ops)
        own.rt = rt
        own._branch(*([part, post] if block is PostNormBlock else [pre, part, post]), stream, None)
        got.append(stream.value())
        if isinstance(rt.ops, GroupedOps):
            assert rt.ops.grouped_calls == (0 if products_only else 1)
    assert (got[0] - got[1]).abs().max() <= 1e-5 * got[1].abs().max()
