"""A prompt's linear with what follows it in one launch (gemm_k64.hip, After): the bits of the separate launches, for both
tiles (as 256 compute units pick them), head sizes, group sizes and kinds of scales, and rows and channels that fill no
tile; and a decoder's prompts with all, some and none of its linears run that way."""
import numpy as np
import pytest


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _case(rng, rows, k, n, group, uniform, bias=True):
    import volvoxai_amd as vx
    from volvoxai_amd.decoder import pack_w8_words
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    scales = rng.uniform(0.002, 0.01, (n, 1)).astype(np.float32).repeat((k + group - 1) // group, 1)
    if not uniform:
        scales = scales * rng.uniform(0.7, 1.0, scales.shape).astype(np.float32)
    pl = vx.PackedLinear(pack_w8_words(w), scales, rng.normal(0, 0.1, n).astype(np.float32) if bias else None, k, n, group)
    a8 = _dev(rng.integers(-127, 128, (rows, k)).astype(np.int8))
    sc = rng.uniform(0.001, 0.01, rows).astype(np.float32)
    sc[rows // 2] = np.nan  # a row that was not finite
    return pl, a8, _dev(sc)


def _same(a, b):
    import torch
    return torch.equal(a.view(torch.int32)[~torch.isnan(a)], b.view(torch.int32)[~torch.isnan(b)]) and torch.equal(torch.isnan(a), torch.isnan(b))


@pytest.mark.gpu
@pytest.mark.parametrize("group,uniform", [(64, True), (64, False), (128, True), (128, False), (256, True)])
@pytest.mark.parametrize("rows,t,q_heads,kv_heads,hd,k,tile", [
    (9, 77, 16, 8, 128, 256, 64), (7, 190, 12, 6, 64, 416, 64), (32, 128, 16, 8, 128, 512, 128), (33, 101, 9, 3, 64, 256, 128),
    (1, 1027, 6, 3, 128, 272, 64), (31, 130, 16, 8, 128, 256, 128), (3, 1201, 21, 3, 64, 256, 128)])
def test_rotary_and_append_behind_the_linear(ctx, rows, t, q_heads, kv_heads, hd, k, tile, group, uniform):
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(rows * t + hd + group)
    max_seq = t + 5
    pl, a8, sc = _case(rng, rows * t, k, (q_heads + 2 * kv_heads) * hd, group, uniform)
    cos, sin = (_dev(rng.normal(0, 1, (max_seq, hd)).astype(np.float32)) for _ in range(2))
    positions = torch.arange(t, device="cuda") + 3
    caches = [torch.full((rows, kv_heads, max_seq, hd), 7.0, device="cuda") for _ in range(4)]
    st, qkv = pl.forward_a8(ctx, a8, sc)
    want = vx.rope_append_kv(ctx, qkv.reshape(rows, t, -1), cos, sin, positions, q_heads, kv_heads, hd, caches[0], caches[1])
    handled, q = pl.rope_append_a8(ctx, a8, sc, t, cos, sin, positions, q_heads, kv_heads, hd, caches[2], caches[3])
    ctx.synchronize()
    assert st == 0 and handled and ctx.last_variant.endswith(f".t{tile}x{tile}k64-rope"), ctx.last_variant
    assert _same(q, want) and _same(caches[2], caches[0]) and _same(caches[3], caches[1])
    # a position past the caches: nothing of that token is touched, and a fault bit says so
    positions[t - 1] = max_seq
    before = caches[2].clone(), caches[3].clone()
    handled, q = pl.rope_append_a8(ctx, a8, sc, t, cos, sin, positions, q_heads, kv_heads, hd, caches[2], caches[3])
    assert handled and ctx.fault_flags() == 4 and _same(caches[2], before[0]) and _same(caches[3], before[1])
    assert _same(q[:, :t - 1], want[:, :t - 1])
    ctx.clear_fault_flags()
    pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("group,uniform", [(64, True), (128, False), (128, True), (256, False)])
@pytest.mark.parametrize("rows,k,inter,tile", [(4096, 256, 3072, 128), (700, 512, 1536, 64), (1300, 272, 1056, 64), (2500, 128, 800, 64),
                                               (2049, 256, 1120, 64), (4001, 256, 3104, 128), (2945, 128, 3104, 128)])
def test_swiglu_and_add_behind_the_linear(ctx, rows, k, inter, tile, group, uniform):
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(rows + k + group)
    pl, a8, sc = _case(rng, rows, k, 2 * inter, group, uniform, bias=rows % 2 == 0)
    st, gu = pl.forward_a8(ctx, a8, sc)
    ctx.synchronize()
    *_, want = vx.swiglu_prepare_i8(ctx, gu, want_activated=True)
    handled, act = pl.swiglu_a8(ctx, a8, sc)
    ctx.synchronize()
    assert st == 0 and handled and ctx.last_variant.endswith(f".t{tile}x{tile}k64-swiglu"), ctx.last_variant
    assert _same(act, want)
    x = _dev(rng.normal(0, 1, (rows, 2 * inter)).astype(np.float32))
    want = x + gu
    assert pl.add_a8(ctx, a8, sc, x)
    ctx.synchronize()
    assert ctx.last_variant.endswith(f".t{tile}x{tile}k64-add") and _same(x, want)
    pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("group,uniform", [(64, True), (128, False), (128, True), (256, False)])
@pytest.mark.parametrize("rows,k,n,tile", [(4001, 256, 6212, 128), (3000, 256, 1028, 128), (2945, 128, 6172, 128), (2049, 256, 2244, 64),
                                           (4001, 128, 1100, 64), (1921, 272, 4124, 64)])
def test_add_of_channels_that_end_inside_a_panel(ctx, rows, k, n, tile, group, uniform):
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(rows + k + group)
    pl, a8, sc = _case(rng, rows, k, n, group, uniform, bias=k != 128)
    st, y = pl.forward_a8(ctx, a8, sc)
    # (a guard behind the rows: a store past the last channel of the last row would show)
    x = _dev(rng.normal(0, 1, rows * n + 64).astype(np.float32))
    want = x.clone()
    want[:rows * n] += y.reshape(-1)
    assert st == 0 and pl.add_a8(ctx, a8, sc, x[:rows * n].view(rows, n))
    ctx.synchronize()
    assert ctx.last_variant.endswith(f".t{tile}x{tile}k64-add") and _same(x, want)
    pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,t,handled", [(32, 128, {"rope_append_a8": 2, "swiglu_a8": 1, "add_a8": 2}),
                                            (8, 64, {"rope_append_a8": 2, "swiglu_a8": 1}), (4, 40, {})])
def test_decoder_prompts_with_and_without(monkeypatch, rows, t, handled):
    """Two layers: of a prompt of 512 tokens the q/k/v and gate/up linears run with what follows them and the narrower
    output and down projections do not.  (Behind the last layer's cache append only each row's last token goes on.)"""
    import torch
    import volvoxai_amd as vx
    from volvoxai_amd.decoder import DecoderConfig, W8A8Decoder, init_weights
    cfg = DecoderConfig(layers=2, vocab=1000)
    dec = W8A8Decoder(cfg, init_weights(cfg, 5), rows)
    prompt = torch.randint(0, cfg.vocab, (rows, t), generator=torch.Generator().manual_seed(t)).cuda()
    counts = {}

    def counting(name):
        run = getattr(vx.PackedLinear, name)

        def counted(*args):
            result = run(*args)
            if result[0] if isinstance(result, tuple) else result:
                counts[name] = counts.get(name, 0) + 1
            return result
        return counted

    results = []
    for followed in (True, False):
        with monkeypatch.context() as m:
            for name, declined in (("rope_append_a8", (False, None)), ("swiglu_a8", (False, None)), ("add_a8", False)):
                m.setattr(vx.PackedLinear, name, counting(name) if followed else lambda *args, declined=declined: declined)
            dec.prefill(prompt)
        torch.cuda.synchronize()
        results.append([x.clone() for x in (dec.last_logits, dec.k_cache, dec.v_cache)])
    assert counts == handled
    for with_, without in zip(*results):
        assert torch.equal(with_.view(torch.int32), without.view(torch.int32))
    dec.close()


@pytest.mark.gpu
def test_what_is_declined(ctx):
    """Few rows, and channels that are not whole pair panels, go by the separate launches; heads that are not the linear's
    channels are refused."""
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(3)
    pl, a8, sc = _case(rng, 64, 256, 512, 128, True)
    assert pl.swiglu_a8(ctx, a8, sc)[0] is False and pl.add_a8(ctx, a8, sc, torch.zeros((64, 512), device="cuda")) is False
    cache = torch.zeros((1, 1, 64, 64), device="cuda")
    table = torch.zeros((64, 64), device="cuda")
    with pytest.raises(RuntimeError):
        pl.rope_append_a8(ctx, a8, sc, 64, table, table, torch.arange(64, device="cuda"), 2, 1, 64, cache, cache)
    pl.close()
    pl, a8, sc = _case(rng, 4096, 128, 2 * 1000, 128, True)
    assert pl.swiglu_a8(ctx, a8, sc)[0] is False
    pl.close()
