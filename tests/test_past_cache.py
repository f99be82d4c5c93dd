"""Weights that steps of few rows read past the last-level cache: which are marked, and that the mark changes no result."""
from types import SimpleNamespace

import pytest
import torch

from machserve_amd.engine.loading import mark_weights_past_cache

DEV = "cuda:0"


def _part(**tensors):
    return SimpleNamespace(parts=None, **tensors)


def _model(blocks, order=None, tied=False):
    w = lambda n: torch.zeros((n, 8), dtype=torch.bfloat16)  # noqa: E731  16 n bytes
    embedding, head = _part(weight=w(1000)), _part(weight=None if tied else w(900))
    made = [SimpleNamespace(parts=lambda ps=ps: ps) for ps in blocks]
    return SimpleNamespace(embedding=embedding, head=head, blocks=made, order=order or list(range(len(made))),
                           rt=SimpleNamespace(dtype=torch.bfloat16), parts=lambda: [embedding, *(p for b in blocks for p in b), head])


def test_the_largest_weights_are_marked_so_that_the_others_fit():
    w = lambda n, dt=torch.bfloat16: torch.zeros((n, 8), dtype=dt)  # noqa: E731
    parts = [_part(a=w(10), b=w(100), v=torch.zeros(64), f=w(4000, torch.float32)), _part(many=[w(20), w(300)])]
    m = _model([parts])
    assert mark_weights_past_cache(m, 16 * 1330) == 0 and not parts[0].b.past_cache
    assert mark_weights_past_cache(m, 16 * 429) == 16 * (300 + 900)
    assert [t.past_cache for t in (parts[0].a, parts[1].many[0], parts[0].b, parts[1].many[1], m.head.weight)] == [False, False, False, True, True]
    assert not hasattr(parts[0].v, "past_cache") and not hasattr(parts[0].f, "past_cache") and not hasattr(m.embedding.weight, "past_cache")
    assert mark_weights_past_cache(m, 16 * 2000) == 0 and not m.head.weight.past_cache  # a mark does not outlive the choice


def test_a_tied_table_is_a_weight_and_a_layer_that_runs_again_is_not_marked():
    w = lambda n: torch.zeros((n, 8), dtype=torch.bfloat16)  # noqa: E731
    once, twice = _part(a=w(500)), _part(a=w(600))
    m = _model([[once], [twice]], order=[0, 1, 1], tied=True)
    assert mark_weights_past_cache(m, 0) == 16 * 1500
    assert m.embedding.weight.past_cache and once.a.past_cache and not hasattr(twice.a, "past_cache")


# every product that reads a marked weight: few rows in one, two and four row tiles, tiles of 64 rows with four buffers, and more rows, where the mark says nothing
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 130])
@pytest.mark.parametrize("N,K", [(96, 256), (1000, 1024), (2048, 5632)])
def test_a_marked_weight_gives_the_same_bits(dtype, M, N, K):
    from machserve_amd.kernels import get_ops
    ops = get_ops(dtype, DEV)
    gen = torch.Generator().manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(s, generator=gen).to(DEV, dtype)  # noqa: E731
    a, w, gu, x = rnd(M, K), rnd(N, K), rnd(2 * 16 * -(-N // 16), K), torch.randn((M, N), generator=gen).to(DEV)
    norm_w = torch.ones(N, device=DEV)

    def products():
        stream = x.clone()
        out = [ops.linear(a, w), ops.linear(a, w, out_f32=True), ops.linear_split(a, w), ops.linear_act(a, w, "silu"), ops.linear_swiglu(a, gu, N),
               ops.linear_residual(a, w, stream), stream]
        if ops.prenorm_swiglu_takes(M, N, K, 2 * N):
            stream = x.clone()
            out += [*ops.linear_residual_prenorm(a, w, stream, norm_w), stream]
        if ops._plan("ms_swiglu_scaled_takes", M, gu.shape[0] // 2, K):
            out.append(ops.linear_swiglu_scaled(a, torch.ones((1, M), device=DEV), 1e-6, gu, gu.shape[0] // 2))
        return out

    plain = products()
    w.past_cache = gu.past_cache = True
    for one, other in zip(plain, products()):
        assert (one is None and other is None) or torch.equal(one, other)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 100])
def test_marked_experts_give_the_same_bits(T):
    from machserve_amd.kernels import get_ops
    ops = get_ops(torch.bfloat16, DEV)
    E, d, ff, shared = 4, 256, 320, 256
    gen = torch.Generator().manual_seed(T)
    rnd = lambda *s: torch.randn(s, generator=gen).to(DEV, torch.bfloat16)  # noqa: E731
    h, router, up, down = rnd(T, d), torch.randn((E, d), generator=gen).to(DEV), rnd(2 * (E * ff + shared), d), rnd(d, E * ff + shared)
    run = lambda: ops.routed_experts(h, router, None, 2, up, down, E, ff, shared, "silu", gated=True)  # noqa: E731
    plain = run()
    up.past_cache = down.past_cache = True
    assert all(torch.equal(p, q) for p, q in zip(plain, run()))


# attention with blocks beside its own that read weights ahead: the 32-row kernel and the general one, whole and cut, one weight and two, of a few bytes, and some that are not taken (too large, beginning anywhere, spread out)
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hd,before,splits", [(64, 0, 0), (64, 900, 3), (128, 0, 0), (96, 0, 0), (96, 900, 2)])
def test_an_attention_that_reads_ahead_gives_the_same_bits(dtype, hd, before, splits):
    from machserve_amd.kernels import get_ops
    ops = get_ops(dtype, DEV)
    T, H, KV, ps = 130, 4, 2, 64
    gen = torch.Generator().manual_seed(hd + before)
    pages = -(-(T + before) // ps)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    q = torch.randn((T, H * hd), generator=gen).to(DEV, dtype)
    kp, vp = torch.randn((pages, KV, ps, hd), generator=gen).to(DEV, dtype), torch.randn((pages, KV, hd, ps), generator=gen).to(DEV, dtype)
    unit = ops.attention_rows_per_block(hd)
    work = i32([[0, r] for r in range(0, T * (H // KV), unit)])
    run = lambda **kw: ops.paged_attention(q, kp, vp, i32([list(range(pages))]), i32([0]), i32([T]), i32([before]), work, H, KV, hd, ps, None,  # noqa: E731
                                           hd ** -0.5, key_splits=splits, **kw)
    plain = run()
    small, odd, wide = (torch.zeros(n, dtype=dtype, device=DEV) for n in (4, 40961, (ops.AHEAD_BYTES >> 1) // plain.element_size()))
    for ahead in ((small,), (odd,), (odd, wide), (wide, wide), (torch.cat([wide, wide, odd]),), (odd[1:], wide[:1].expand(1 << 24))):
        assert torch.equal(run(ahead=ahead), plain)


def test_what_a_mixer_reads_ahead_is_its_feed_forward():
    from machserve_amd.engine.loading import mark_weights_ahead
    from machserve_amd.parts.base import Mixer
    w = lambda n, dt=torch.bfloat16: torch.zeros((n, 8), dtype=dt)  # noqa: E731
    inner, mixer = Mixer.__new__(Mixer), Mixer.__new__(Mixer)
    mixer.sub_parts = lambda: [inner]
    up, down = w(200), w(90)
    blocks = [SimpleNamespace(feed_forward=SimpleNamespace(up=up, down=down, router=w(4, torch.float32), bias=torch.zeros(8, dtype=torch.bfloat16)), mixers=lambda: [mixer]),
              SimpleNamespace(feed_forward=None, mixers=lambda: [Mixer.__new__(Mixer)])]
    model = SimpleNamespace(blocks=blocks, rt=SimpleNamespace(dtype=torch.bfloat16, ops=object()))
    mark_weights_ahead(model)
    assert mixer.ahead == () and mixer.reading_ahead() == {}  # stand-ins for the kernels take no such argument
    model.rt.ops = SimpleNamespace(AHEAD_BYTES=1)
    mark_weights_ahead(model)
    assert [t is want for t, want in zip(mixer.ahead, (down, up))] == [True, True] and inner.ahead == mixer.ahead and inner.reading_ahead() == {"ahead": inner.ahead}
