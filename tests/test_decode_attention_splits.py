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
