"""Rotary embedding and cache append in 16-byte chunks: head sizes, remainders and operands the chunks do not take."""
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
@pytest.mark.parametrize("q_heads,kv_heads,head_dim,offset", [
    (16, 8, 128, 0), (8, 4, 64, 0),   # two chunks a thread; fewer than the smaller workgroup
    (3, 1, 8, 0), (2, 1, 1024, 0),    # the smallest and the largest head of 16-byte chunks
    (5, 5, 256, 0), (9, 1, 16, 0),    # chunks that fill no whole round
    (4, 2, 96, 0), (4, 2, 128, 1),    # a head size that is no power of two; operands off their 16 bytes
])
def test_rope_append_chunks(ctx, q_heads, kv_heads, head_dim, offset):
    """Two products and one sum per channel, each rounded: the same bits as numpy's f32."""
    import torch
    from volvoxai_amd import w8a8
    rng = np.random.default_rng(head_dim + offset)
    rows, t, max_seq = 3, 5, 11
    shape = (rows, t, q_heads + 2 * kv_heads, head_dim)
    qkv = rng.normal(0, 1, shape).astype(np.float32)
    cos, sin = (rng.normal(0, 1, (max_seq, head_dim)).astype(np.float32) for _ in range(2))
    positions = np.array([3, 10, 0, 4, 7], np.int64)
    flat = torch.zeros(qkv.size + offset, device="cuda")
    flat[offset:] = torch.from_numpy(qkv.reshape(-1)).cuda()
    k, v = (torch.full((rows, kv_heads, max_seq, head_dim), 9.0, device="cuda") for _ in range(2))
    q = w8a8.rope_append_kv(ctx, flat[offset:].view(rows, t, -1), torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda(),
                            torch.from_numpy(positions).cuda(), q_heads, kv_heads, head_dim, k, v)
    ctx.synchronize()
    half = head_dim // 2
    turned = np.concatenate([-qkv[..., half:], qkv[..., :half]], -1)
    c, s = cos[positions][None, :, None], sin[positions][None, :, None]
    want = qkv * c + turned * s
    keys, values = (np.full((rows, kv_heads, max_seq, head_dim), 9.0, np.float32) for _ in range(2))
    keys[:, :, positions] = want[:, :, q_heads:q_heads + kv_heads].transpose(0, 2, 1, 3)
    values[:, :, positions] = qkv[:, :, q_heads + kv_heads:].transpose(0, 2, 1, 3)
    assert (q.cpu().numpy().reshape(rows, t, q_heads, head_dim) == want[:, :, :q_heads]).all()
    assert (k.cpu().numpy() == keys).all() and (v.cpu().numpy() == values).all()
