"""Decode attention at head sizes 64 and 128: one walk over keys and values, blocks of 256 slots, eight wavefronts that take eight
slots of every 64 each, and four query heads a workgroup by way of scores in LDS at head size 128."""
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
@pytest.mark.parametrize("position", [0, 1, 7, 16, 127, 128, 144, 255, 256, 300, 511, 519])
@pytest.mark.parametrize("rows,q_heads,kv_heads,head_dim", [
    (1, 4, 2, 128), (1, 2, 2, 64),        # one query head a workgroup
    (40, 8, 4, 128), (40, 8, 4, 64),      # two
    (20, 16, 2, 128), (20, 16, 1, 64),    # four
])
def test_decode_attention_blocks(ctx, rows, q_heads, kv_heads, head_dim, position):
    """Against the definition in float64, the fused launch and the plain one with the same bits; slots behind the
    token's own hold NaN.  (f32 dots of head_dim products: about 1e-6 relative per probability.)"""
    import torch
    from volvoxai_amd import w8a8
    rng = np.random.default_rng(position * 7 + rows)
    max_seq, rep = 520, q_heads // kv_heads
    qkv = rng.normal(0, 1, (rows, 1, (q_heads + 2 * kv_heads) * head_dim)).astype(np.float32)
    cache = rng.normal(0, 1, (2, rows, kv_heads, max_seq, head_dim)).astype(np.float32)
    cache[:, :, :, position:] = np.nan
    if position > 2:
        cache[0, 0, 0, 2] *= 30.0  # one slot takes most of the weight: maxima jump, groups differ
        cache[0, 0, 0, 1, 0] = -np.inf  # (a score of -inf or +inf, by the query's sign: nothing, or NaN)
    angle = rng.uniform(0, 6.28, (max_seq, head_dim)).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()
    cos, sin, x, pos = dev(np.cos(angle)), dev(np.sin(angle)), dev(qkv), torch.tensor([position], device="cuda")
    k1, v1, k2, v2 = dev(cache[0]), dev(cache[1]), dev(cache[0]), dev(cache[1])
    q = w8a8.rope_append_kv(ctx, x, cos, sin, pos, q_heads, kv_heads, head_dim, k1, v1)
    plain = w8a8.gqa_attention(ctx, q, k1, v1, pos).reshape(rows, q_heads, head_dim)
    fused = w8a8.rope_gqa_attention_decode(ctx, x.reshape(rows, -1), cos, sin, pos, q_heads, kv_heads, head_dim, k2, v2)
    ctx.synchronize()
    assert torch.equal(plain.reshape(rows, -1).view(torch.int32), fused.view(torch.int32))
    k, v = (a.cpu().numpy()[:, :, :position + 1].astype(np.float64) for a in (k2, v2))
    assert np.array_equal(k2.cpu().numpy(), k1.cpu().numpy(), equal_nan=True)
    assert np.array_equal(v2.cpu().numpy(), v1.cpu().numpy(), equal_nan=True)
    q = q.cpu().numpy().reshape(rows, q_heads, head_dim).astype(np.float64)
    got = plain.cpu().numpy()
    with np.errstate(invalid="ignore"):
        for h in range(q_heads):
            sc = np.matmul(k[:, h // rep], q[:, h, :, None])[:, :, 0] / np.sqrt(head_dim)
            p = np.exp(sc - sc.max(-1, keepdims=True))
            want = np.matmul((p / p.sum(-1, keepdims=True))[:, None], v[:, h // rep])[:, 0]
            # (a score of the strong slot is up to about 150: its f32 rounding is 1e-5 of a probability)
            assert np.allclose(got[:, h], want, rtol=2e-5, atol=1e-4 if h < rep else 5e-6, equal_nan=True), h
