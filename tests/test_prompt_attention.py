"""The matrix-pipe prompt attention (head sizes 64 and 128) at the edges of its tiles: 32 queries a wavefront, 32
slots a tile, a workgroup's wavefronts on neighbouring tokens (many query blocks, or at most 32 tokens) or sharing
their queries (few)."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def ctx():
    import torch
    import volvoxai_amd as vx
    c = vx.Context(0, torch.cuda.current_stream())
    yield c
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,t,start,q_heads,kv_heads,head_dim,max_seq,order", [
    (128, 33, 0, 16, 8, 128, 33, "rising"),     # neighbouring tokens: ragged last block and last group of four
    (64, 97, 7, 16, 16, 64, 111, "rising"),     # the same at head size 64, a full cache but for the last slots
    (1, 33, 0, 2, 1, 128, 65, "rising"),        # shared queries: a second tile of one slot, wavefronts without a tile
    (2, 64, 64, 8, 4, 64, 160, "rising"),       # the same at head size 64: whole tiles, a prompt continued
    (1, 129, 60, 32, 1, 128, 190, "rising"),    # 32 query heads per KV head: one token a wavefront
    (3, 32, 1, 6, 2, 64, 34, "rising"),         # three heads per KV head: 30 of 32 queries
    (2, 8, 0, 4, 2, 128, 16, "rising"),         # fewest tokens of the path
    (2, 45, 3, 4, 2, 128, 60, "shuffled"),      # positions in any order: no wavefront's span follows from its place
])
def test_prompt_attention_tiles(ctx, rows, t, start, q_heads, kv_heads, head_dim, max_seq, order):
    """Against the definition in float64; cache slots no token sees hold NaN.  A score is head_dim products of about
    unit variance summed in f32 (error about 1e-6), which is the relative error of its probability."""
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(rows * 1000 + t)
    q = rng.normal(0, 1, (rows, t, q_heads, head_dim)).astype(np.float32)
    k = rng.normal(0, 1, (rows, kv_heads, max_seq, head_dim)).astype(np.float32)
    v = rng.normal(0, 1, (rows, kv_heads, max_seq, head_dim)).astype(np.float32)
    positions = np.arange(start, start + t, dtype=np.int64)
    if order == "shuffled":
        positions = rng.permutation(positions)
    k[:, :, start + t:] = np.nan
    v[:, :, start + t:] = np.nan
    k[0, 0, start + 2, :] *= 40.0  # one slot takes most of the weight: the running maximum jumps
    out = vx.gqa_attention(ctx, *(torch.from_numpy(a).cuda() for a in (q, k, v, positions)))
    ctx.synchronize()
    got = out.cpu().numpy().reshape(rows, t, q_heads, head_dim)
    seen, rep = start + t, q_heads // kv_heads
    hidden = np.arange(seen)[None, :] > positions[:, None]
    for h in range(q_heads):
        kk, vv = (a[:, h // rep, :seen].astype(np.float64) for a in (k, v))
        sc = np.matmul(q[:, :, h].astype(np.float64), kk.transpose(0, 2, 1)) / np.sqrt(head_dim)
        sc[:, hidden] = -np.inf
        p = np.exp(sc - sc.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        # (a score of the strong slot is up to about 200: its f32 rounding is 1e-5 of a probability)
        assert np.allclose(got[:, :, h], np.matmul(p, vv), rtol=2e-5, atol=1e-4 if h < rep else 5e-6), h


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,t", [(128, 20), (128, 70), (64, 70)])
def test_prompt_attention_of_infinite_scores(ctx, head_dim, t):
    """Scores of -inf count nothing, also where a whole first tile has no other; a NaN or +inf score makes its row NaN."""
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(t)
    q = np.ones((1, t, 1, head_dim), np.float32)
    k = np.zeros((1, 1, 96, head_dim), np.float32)
    v = rng.normal(0, 1, (1, 1, 96, head_dim)).astype(np.float32)
    low, bad = (32, 50) if t > 60 else (5, 12)
    k[0, 0, :low, 0] = -np.inf
    k[0, 0, bad, 0] = np.inf
    positions = np.arange(t, dtype=np.int64)
    out = vx.gqa_attention(ctx, *(torch.from_numpy(a).cuda() for a in (q, k, v, positions)))
    ctx.synchronize()
    got = out.cpu().numpy().reshape(t, head_dim)
    assert np.isnan(got[:low]).all() and np.isnan(got[bad:]).all()  # (nothing but -inf: 0 / 0, as exp(-inf + inf) gives)
    for i in range(low, bad):
        assert np.allclose(got[i], v[0, 0, low:i + 1].astype(np.float64).mean(0), rtol=1e-5, atol=1e-6), i


@pytest.mark.gpu
@pytest.mark.parametrize("q_heads,max_seq,taken", [(1, 30000, True), (1, 40000, False), (8, 14000, True), (8, 15000, False)])
def test_prompt_attention_cache_limits(ctx, q_heads, max_seq, taken):
    """The longest caches are those whose score rows fit one of the kernels that keep them, whichever kernel answers."""
    import torch
    import volvoxai_amd.w8a8 as vx
    q = torch.randn(1, 8, q_heads, 64, device="cuda")
    k, v = torch.randn(2, 1, 1, max_seq, 64, device="cuda")
    positions = torch.arange(max_seq - 8, max_seq, device="cuda")
    if not taken:
        with pytest.raises(vx.VxHipError):
            vx.gqa_attention(ctx, q, k, v, positions)
        return
    out = vx.gqa_attention(ctx, q, k, v, positions).reshape(8, q_heads, 64)
    ctx.synchronize()
    scores = torch.matmul(q[0].double(), k[0, 0].double().T) / 8.0  # [t, heads, slots]
    scores.masked_fill_(torch.arange(max_seq, device="cuda")[None, None] > positions[:, None, None], float("-inf"))
    want = torch.matmul(torch.softmax(scores, -1), v[0, 0].double())
    # (30,000 terms summed in f32: each adds at most 2^-24 of a sum of probabilities times values below 1)
    assert torch.allclose(out.double(), want, rtol=2e-5, atol=5e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,t,layers,q_heads,kv_heads,head_dim,max_seq", [
    (1, 9, 1, 2, 2, 128, 14300),      # one row: the score buffer of the decode kernel would be too small
    (17, 8, 1, 16, 8, 128, 6600),     # more query heads than compute units: two heads share that buffer
    (1, 40, 2, 2, 2, 64, 14900),
    (3, 5, 1, 4, 2, 64, 40),          # fewer tokens than the prompt kernels take
    (2, 37, 1, 4, 2, 128, 40),
])
def test_decoder_prompts_behind_the_last_layer(oracle, rows, t, layers, q_heads, kv_heads, head_dim, max_seq):
    """Behind the last layer only each row's last token is computed: the CPU restatement's logits, for every cache that
    the layers in front take, and the same bits whatever its length.  (An activation next to a rounding boundary may
    take the neighbouring code, one of 127: the logits then differ by less than 1 / 127 of their norm.)"""
    import torch
    from _decoder_ref import DecoderRef
    from volvoxai_amd.decoder import DecoderConfig, W8A8Decoder, init_weights, rope_tables
    sizes = dict(layers=layers, hidden=256, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, inter=256, vocab=300)
    cfg, short = DecoderConfig(max_seq=max_seq, **sizes), DecoderConfig(max_seq=48, **sizes)
    weights = init_weights(short, 3)
    prompt = np.random.default_rng(t).integers(0, cfg.vocab, (rows, t))
    ref = DecoderRef(short, weights, oracle, rope_tables)
    empty = [[np.zeros((rows, kv_heads, 0, head_dim), np.float32) for _ in range(layers)] for _ in range(2)]
    want = ref.forward(prompt, 0, *empty)
    logits = []
    for c in (short, cfg):
        dec = W8A8Decoder(c, weights, rows)
        torch.cuda.synchronize()
        dec.prefill(torch.from_numpy(prompt).cuda())
        logits.append(dec.last_logits.cpu().numpy())
        dec.close()
    assert (logits[0].view(np.uint32) == logits[1].view(np.uint32)).all()
    assert np.linalg.norm(logits[1] - want) <= np.linalg.norm(want) / 127


@pytest.mark.gpu
@pytest.mark.parametrize("rows,head_dim,t", [(1, 128, 20), (1, 128, 70), (64, 64, 70), (1, 64, 70), (1, 64, 1), (1, 64, 3)])
def test_values_at_the_ends_of_the_range(ctx, rows, head_dim, t):
    """A value that is not finite reaches the tokens that see its slot and no others; values near the largest f32 leave
    a mean of their size (probabilities of one sum to one within 2^-18 here)."""
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(t)
    q = rng.normal(0, 1, (rows, t, 2, head_dim)).astype(np.float32)
    k = rng.normal(0, 1, (rows, 1, 96, head_dim)).astype(np.float32)
    v = rng.normal(0, 1, (rows, 1, 96, head_dim)).astype(np.float32)
    start = 96 - t if t < 8 else 0
    positions = np.arange(start, start + t, dtype=np.int64)
    nan, inf = start + t // 2, start + t - t // 4
    v[:, 0, nan, 3] = np.nan
    if inf < start + t:
        v[:, 0, inf, 5] = -np.inf
    sc = np.matmul(q.transpose(0, 2, 1, 3).astype(np.float64), k.transpose(0, 1, 3, 2)) / np.sqrt(head_dim)
    dev = lambda a: torch.from_numpy(a).cuda()
    got = vx.gqa_attention(ctx, dev(q), dev(k), dev(v), dev(positions)).reshape(rows, t, 2, head_dim)
    big = vx.gqa_attention(ctx, dev(q), dev(k), torch.full((rows, 1, 96, head_dim), 3.3e38, device="cuda"), dev(positions))
    ctx.synchronize()
    got = got.cpu().numpy()
    for i in range(t):
        seen = sc[:, :, i, :positions[i] + 1]
        p = np.exp(seen - seen.max(-1, keepdims=True))
        with np.errstate(invalid="ignore"):
            want = np.matmul(p / p.sum(-1, keepdims=True), v[:, 0, :positions[i] + 1].astype(np.float64))
        assert np.allclose(got[:, i], want, rtol=2e-5, atol=5e-6, equal_nan=True), i
    assert torch.allclose(big.double(), torch.full_like(big, 3.3e38).double(), rtol=2.0 ** -18, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 3.0])
@pytest.mark.parametrize("rows,head_dim", [(2, 64), (2, 128), (40, 64), (40, 128)])
def test_prompt_attention_error_against_float64(ctx, rows, head_dim, scale):
    """No further from float64 than dots summed in f32 in chains of 64 channels (fused multiply-adds), a softmax in f32 and
    values summed slot by slot.  (65,536 outputs and more: the ratio of the two errors' norms varies by about 1 %
    from draw to draw, and a single chain of 128 channels has 1.4 times the error.)"""
    import torch
    import volvoxai_amd.w8a8 as vx
    t, heads = 128, 4
    gen = torch.Generator(device="cuda").manual_seed(head_dim + rows)
    q = torch.randn((rows, t, heads, head_dim), generator=gen, device="cuda") * scale
    k = torch.randn((rows, heads, t, head_dim), generator=gen, device="cuda")
    v = torch.randn((rows, heads, t, head_dim), generator=gen, device="cuda")
    positions = torch.arange(t, device="cuda")
    got = vx.gqa_attention(ctx, q, k, v, positions).reshape(rows, t, heads, head_dim).transpose(1, 2).double()
    ctx.synchronize()
    qt, hidden = q.transpose(1, 2).contiguous(), positions[None, :] > positions[:, None]
    fma = lambda s, a, b: (s.double() + a.double() * b.double()).float()
    dots = []
    for c0 in range(0, head_dim, 64):
        s = torch.zeros((rows, heads, t, t), device="cuda")
        for c in range(c0, c0 + 64):
            s = fma(s, qt[..., c, None], k[:, :, None, :, c])
        dots.append(s)
    inverse = float(np.float32(1.0 / np.sqrt(head_dim)))
    p = torch.softmax((sum(dots) * inverse).masked_fill(hidden, float("-inf")), -1)
    held = torch.zeros((rows, heads, t, head_dim), device="cuda")
    for s in range(t):
        held = fma(held, p[..., s, None], v[:, :, None, s])
    exact = torch.zeros((rows, heads, t, t), device="cuda", dtype=torch.float64)
    for c in range(head_dim):
        exact += qt[..., c, None].double() * k[:, :, None, :, c].double()
    p64 = torch.softmax((exact / np.sqrt(head_dim)).masked_fill(hidden, float("-inf")), -1)
    want = sum(p64[..., s, None] * v[:, :, None, s].double() for s in range(t))
    error, held_error = (got - want).norm().item(), (held.double() - want).norm().item()
    assert error <= 1.1 * held_error, error / held_error
