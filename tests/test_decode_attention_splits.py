"""Decode attention at head sizes 64 and 128: each way a launch is split (a head on four workgroups, on two, on one, two and four
heads a workgroup), with positions at the ends of its strips of eight slots, rounds of 64 and blocks of 256."""
import pytest
import test_decode_attention as blocks
from test_decode_attention import ctx  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("position", [0, 7, 8, 63, 64, 199, 255, 256, 263, 512])
@pytest.mark.parametrize("rows,q_heads,kv_heads,head_dim", [
    (3, 8, 4, 128), (7, 16, 8, 128), (9, 16, 8, 128),  # a head on four, two; two heads on one
    (50, 3, 1, 128), (33, 8, 8, 128),                  # a head a workgroup, its rows read by three or by one
    (130, 8, 1, 128),                                  # four heads a workgroup, by way of scores in LDS
    (5, 8, 4, 64), (24, 8, 4, 64), (90, 3, 1, 64),     # a head on two, on one
    (65, 8, 4, 64), (130, 8, 1, 64),                   # two and four heads a workgroup
    (20, 32, 4, 64), (33, 16, 4, 64),                  # four from two heads a compute unit on
    (20, 32, 4, 128),                                  # by way of scores in LDS, the cache longer than 256 slots
])
def test_decode_attention_splits(ctx, rows, q_heads, kv_heads, head_dim, position):  # noqa: F811
    blocks.test_decode_attention_blocks(ctx, rows, q_heads, kv_heads, head_dim, position)


@pytest.mark.gpu
@pytest.mark.parametrize("position", [256, 319, 320, 383, 384, 447, 448, 511, 512, 519])
@pytest.mark.parametrize("rows,q_heads,kv_heads,head_dim", [(3, 8, 4, 128), (9, 16, 8, 128), (50, 3, 1, 128), (5, 8, 4, 64), (65, 8, 4, 64), (130, 8, 1, 64)])
def test_first_blocks_that_are_not_whole(ctx, rows, q_heads, kv_heads, head_dim, position):  # noqa: F811
    """Past 256 slots: one to four rounds of 64 in the first block, the last round with strips of one wavefront and of all, two
    blocks and three."""
    blocks.test_decode_attention_blocks(ctx, rows, q_heads, kv_heads, head_dim, position)


@pytest.mark.gpu
@pytest.mark.parametrize("position", [200, 300])
@pytest.mark.parametrize("rows,q_heads,kv_heads,head_dim", [
    (24, 24, 8, 128), (96, 6, 2, 128), (24, 32, 8, 128),  # KV heads first, rows first, two heads a workgroup
    (70, 6, 2, 128), (64, 10, 2, 64),                     # neither; rows first
])
def test_workgroups_of_a_kv_head_side_by_side(ctx, rows, q_heads, kv_heads, head_dim, position):  # noqa: F811
    """Launches of one and a half workgroups a compute unit and more whose KV heads have several."""
    blocks.test_decode_attention_blocks(ctx, rows, q_heads, kv_heads, head_dim, position)


@pytest.mark.gpu
@pytest.mark.parametrize("first", [0, 250])
@pytest.mark.parametrize("rows,t,q_heads,kv_heads,head_dim", [(3, 5, 16, 8, 128), (8, 3, 8, 4, 128), (16, 2, 4, 4, 64), (40, 7, 3, 1, 128), (3, 7, 8, 4, 64)])
def test_several_tokens_a_row(ctx, rows, t, q_heads, kv_heads, head_dim, first):  # noqa: F811
    """Two to seven tokens a row, KV heads or rows first where there are eight of them: the bits of a launch a token."""
    import torch
    from volvoxai_amd import w8a8
    gen = torch.Generator(device="cuda").manual_seed(rows * t)
    k, v = (torch.randn((rows, kv_heads, 264, head_dim), device="cuda", generator=gen) for _ in range(2))
    q = torch.randn((rows, t, q_heads, head_dim), device="cuda", generator=gen)
    positions = torch.arange(first, first + t, device="cuda")
    together = w8a8.gqa_attention(ctx, q, k, v, positions)
    apart = [w8a8.gqa_attention(ctx, q[:, i:i + 1].contiguous(), k, v, positions[i:i + 1]) for i in range(t)]
    ctx.synchronize()
    assert torch.equal(together.reshape(rows, t, -1).view(torch.int32), torch.cat([a.reshape(rows, 1, -1) for a in apart], 1).view(torch.int32))


@pytest.mark.gpu
def test_query_heads_that_share_their_rows():
    """32 rows of 2000 slots of 8 KV heads are 526 MB, more than any cache of the device: 32 query heads, on two workgroups a KV head,
    read them once like 16 heads on one (a fifth slower; twice as slow while each of the two read for itself)."""
    import torch
    import volvoxai_amd as vx
    from volvoxai_amd import w8a8
    rows, kv_heads, max_seq, head_dim = 32, 8, 2008, 128
    context = vx.Context(0, torch.cuda.current_stream())
    k, v = (torch.randn((rows, kv_heads, max_seq, head_dim), device="cuda") for _ in range(2))
    table = torch.rand((max_seq, head_dim), device="cuda")
    position = torch.tensor([2000], device="cuda")
    best = {}
    for q_heads in (16, 32):
        qkv = torch.randn((rows, (q_heads + 2 * kv_heads) * head_dim), device="cuda")
        best[q_heads] = 1e9
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                w8a8.rope_gqa_attention_decode(context, qkv, table, table, position, q_heads, kv_heads, head_dim, k, v)
            end.record()
            torch.cuda.synchronize()
            best[q_heads] = min(best[q_heads], start.elapsed_time(end))
    context.close()
    assert best[32] < 1.6 * best[16], best
