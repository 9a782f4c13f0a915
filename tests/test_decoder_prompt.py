"""A prompt as one call (vxhip_decoder_prompt) against the same launches made one by one: the same bits of logits, caches and ids."""
import ctypes as C

import pytest


def _decoder(rows, cfg, seed):
    from volvoxai_amd.decoder import W8A8Decoder, init_weights
    return W8A8Decoder(cfg, init_weights(cfg, seed), rows)


def _one_by_one(dec, tokens):
    """The separate launches, without the linears that take what follows them (the same bits, tests/test_prompt_followed.py)."""
    import torch
    from volvoxai_amd import w8a8 as vx
    cfg, (rows, t) = dec.cfg, tokens.shape
    positions = dec.slots[:t]

    def linear(pl, a8, sc):
        st, y = pl.forward_a8(dec.ctx, a8, sc)
        assert st == 0
        return y

    def norm(x, delta, gain):
        return vx.rmsnorm_prepare_i8(dec.ctx, x, gain, cfg.eps) if delta is None else vx.add_rmsnorm_prepare_i8(dec.ctx, x, delta, gain, cfg.eps)

    x, delta = vx.embedding_gather(dec.ctx, tokens.reshape(-1), dec.embedding), None
    k_cache, v_cache = torch.zeros_like(dec.k_cache), torch.zeros_like(dec.v_cache)
    for li, L in enumerate(dec.layers):
        qkv = linear(L["qkv"], *norm(x, delta, L["gain1"])).reshape(rows, t, -1)
        q = vx.rope_append_kv(dec.ctx, qkv, dec.cos, dec.sin, positions, cfg.q_heads, cfg.kv_heads, cfg.head_dim, k_cache[li], v_cache[li])
        seen = t
        if li == cfg.layers - 1:
            seen = 8 if t >= 8 else 1
        attn = vx.gqa_attention(dec.ctx, q[:, -seen:].contiguous(), k_cache[li], v_cache[li], positions[-seen:])
        if li == cfg.layers - 1:
            x, attn = x.reshape(rows, t, -1)[:, -1].contiguous(), attn[:, -1].contiguous()
        st, o = L["o"].forward_f32(dec.ctx, attn.reshape(-1, cfg.q_dim))
        assert st == 0
        a8, sc = norm(x, o, L["gain2"])
        delta = linear(L["down"], *vx.swiglu_prepare_i8(dec.ctx, linear(L["gate_up"], a8, sc)))
    logits = linear(dec.lm_head, *norm(x, delta, dec.gain_f))
    return logits, vx.argmax_rows(dec.ctx, logits), k_cache, v_cache


@pytest.mark.gpu
@pytest.mark.parametrize("rows,t,layers", [(1, 2, 1), (3, 7, 2), (2, 8, 2), (1, 9, 3), (5, 33, 2), (32, 64, 2)])
@pytest.mark.parametrize("hidden,head_dim", [(512, 64), (258, 36), (1024, 128)])
def test_same_bits_as_the_separate_launches(rows, t, layers, hidden, head_dim):
    """Prompts on both sides of eight tokens, of 32 rows of operand order and of the linears that are followed; widths that are no
    multiple of four floats; a workspace that is used again."""
    import torch
    from volvoxai_amd.decoder import DecoderConfig
    cfg = DecoderConfig(layers=layers, hidden=hidden, q_heads=8, kv_heads=4, head_dim=head_dim, inter=1536, vocab=1000, max_seq=96)
    dec = _decoder(rows, cfg, rows + t)
    try:
        for seed in (1, 2):
            ids = torch.randint(0, cfg.vocab, (rows, t), generator=torch.Generator().manual_seed(seed)).cuda()
            torch.cuda.synchronize()
            with torch.cuda.stream(dec.stream):
                logits, following, k_cache, v_cache = _one_by_one(dec, ids.to(torch.int32))
            dec.k_cache.zero_(), dec.v_cache.zero_()
            torch.cuda.synchronize()
            got = dec.prefill(ids)
            torch.cuda.synchronize()
            assert torch.equal(dec.last_logits.view(torch.int32), logits.view(torch.int32)) and torch.equal(got, following)
            assert torch.equal(dec.k_cache.view(torch.int32), k_cache.view(torch.int32))
            assert torch.equal(dec.v_cache.view(torch.int32), v_cache.view(torch.int32))
    finally:
        dec.close()


@pytest.mark.gpu
def test_refusals():
    """A prompt past the caches, one of another number of rows, a closed linear: errors with nothing launched."""
    import torch
    from volvoxai_amd.decoder import DecoderConfig
    cfg = DecoderConfig(layers=1, hidden=256, q_heads=4, kv_heads=2, head_dim=64, inter=512, vocab=100, max_seq=16)
    dec = _decoder(2, cfg, 3)
    ids = torch.zeros((2, 17), dtype=torch.int64, device="cuda")
    with pytest.raises(ValueError, match="positions"):
        dec.prefill(ids)
    with pytest.raises(ValueError, match="k_cache"):
        dec.prefill(ids[:1, :4])
    dec.prefill(ids[:, :16])
    dec.lm_head.close()
    before = dec.k_cache.clone()
    with pytest.raises(RuntimeError, match="vxhip_decoder_prompt"):
        dec.prefill(ids[:, :8] + 1)
    torch.cuda.synchronize()
    assert torch.equal(before, dec.k_cache)
    dec.close()


@pytest.mark.gpu
@pytest.mark.parametrize("t,changes", [(5, dict(max_seq=16384)), (4, dict(head_dim=128, max_seq=16384)), (9, dict(head_dim=6)), (9, dict(hidden=15364)),
                                       (9, dict(inter=15364)), (9, dict(head_dim=128, q_heads=8, kv_heads=4, max_seq=20000))])
def test_what_a_step_would_refuse_is_refused_before_the_first(t, changes):
    """Caches past the per-token attention's scores and past the prompt's, head sizes and rows that no step takes: an error, and the caches
    are as they were."""
    import torch
    from volvoxai_amd.decoder import DecoderConfig
    cfg = DecoderConfig(**{**dict(layers=2, hidden=64, q_heads=4, kv_heads=2, head_dim=64, inter=96, vocab=50, max_seq=16), **changes})
    dec = _decoder(1, cfg, 3)
    try:
        dec.k_cache.fill_(3.0), dec.v_cache.fill_(3.0)
        torch.cuda.synchronize()
        with pytest.raises(RuntimeError, match="vxhip_decoder_prompt"):
            dec.prefill(torch.zeros((1, t), dtype=torch.int64, device="cuda"))
        torch.cuda.synchronize()
        assert bool((dec.k_cache == 3.0).all()) and bool((dec.v_cache == 3.0).all())
    finally:
        dec.close()


@pytest.mark.gpu
@pytest.mark.parametrize("layers,t,max_seq", [(2, 9, 16384), (1, 5, 14000), (2, 5, 14000)])
def test_long_caches_that_are_taken(layers, t, max_seq):
    """The longest caches of a prompt of eight tokens and more, and of fewer, go on being taken."""
    import torch
    from volvoxai_amd.decoder import DecoderConfig
    cfg = DecoderConfig(layers=layers, hidden=64, q_heads=4, kv_heads=2, head_dim=64, inter=96, vocab=50, max_seq=max_seq)
    dec = _decoder(1, cfg, 3)
    try:
        ids = torch.randint(0, 50, (1, t), generator=torch.Generator().manual_seed(t)).cuda()
        torch.cuda.synchronize()
        with torch.cuda.stream(dec.stream):
            logits, _, _, _ = _one_by_one(dec, ids.to(torch.int32))
        torch.cuda.synchronize()
        dec.prefill(ids)
        torch.cuda.synchronize()
        assert torch.equal(dec.last_logits.view(torch.int32), logits.view(torch.int32))
    finally:
        dec.close()


def test_null_arguments_without_a_device():
    from volvoxai_amd._lib import library
    from volvoxai_amd.w8a8 import _DecoderPrompt
    lib = library()
    assert lib.vxhip_decoder_prompt_workspace(None, None) == 0
    assert lib.vxhip_decoder_prompt_workspace(None, C.byref(_DecoderPrompt())) == 0
    assert lib.vxhip_decoder_prompt(None, C.byref(_DecoderPrompt())) == -1


def test_structures_as_the_header_lays_them_out():
    """Offsets of an LP64 compiler for the header's two structures."""
    from volvoxai_amd.w8a8 import _DecoderLayer, _DecoderPrompt
    assert C.sizeof(_DecoderLayer) == 64 and C.sizeof(_DecoderPrompt) == 144
    assert (_DecoderPrompt.workspace_bytes.offset, _DecoderPrompt.logits.offset, _DecoderPrompt.eps.offset,
            _DecoderPrompt.layer_count.offset, _DecoderPrompt.max_seq.offset) == (72, 80, 96, 104, 136)


@pytest.mark.gpu
def test_fault_words_of_many_contexts():
    """More contexts than the pinned page has lines, destroyed and created again: every one reads its own fault word."""
    import torch
    from volvoxai_amd import w8a8 as vx
    table = torch.ones((4, 8), device="cuda")
    good, bad = torch.tensor([1], dtype=torch.int32, device="cuda"), torch.tensor([9], dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    contexts = [vx.Context(0, None) for _ in range(70)]
    for turn in range(2):
        for i, context in enumerate(contexts):
            vx.embedding_gather(context, bad if i % 3 == turn else good, table, out=torch.empty((1, 8), device="cuda"))
        assert [c.fault_flags() for c in contexts] == [2 if i % 3 == turn else 0 for i in range(70)]
        for c in contexts[::2]:
            c.close()
        for c in contexts[1::2]:
            c.clear_fault_flags()
        contexts[::2] = [vx.Context(0, None) for _ in range(35)]
    for c in contexts:
        c.close()
