"""The narrow tiles of the dequantizing GEMM (gemm_k64.hip) at the edges of their rows, channels and k-blocks."""
import numpy as np
import pytest

import _cases as cases


@pytest.mark.gpu
@pytest.mark.parametrize("grouped", [True, False])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("rows,k,n", [(33, 31, 5), (64, 32, 64), (65, 128, 65), (33, 129, 31), (129, 161, 130), (47, 640, 257),
                                      (96, 1153, 34), (257, 2050, 300)])
def test_narrow_tiles_at_their_edges(ctx, oracle, rows, k, n, group, bits, grouped):
    """One k-block and many, a last k-block with one to four groups of 32, rows and channels that end inside a tile, one
    scale per channel and a scale per group: the oracle's bits, on every tile and on the one the rule picks."""
    import torch
    import volvoxai_amd as vx
    c = cases.packed_case(rows, k, n, group, rows + k + n + bits, True, special_rows=rows == 47)
    scales = c["scales"] if grouped else np.ascontiguousarray(np.broadcast_to(c["scales"][:, :1], c["scales"].shape))
    w = c["w"] if bits == 8 else cases.four_bit(c["w"])
    words = oracle.pack_w8_words(w) if bits == 8 else oracle.pack_w4_words(w)
    _, want = oracle.packed_linear(c["x"], words, scales, c["bias"], n, group, bits=bits)
    pl = vx.PackedLinear(words, scales, c["bias"], k, n, group, weight_bits=bits)
    x = torch.from_numpy(c["x"]).cuda()
    seen = set()
    try:
        for force in (None, "a8-mfma.t64x64k64", "a8-mfma.t64x32k64", "a8-mfma.t32x32k64"):
            vx.force_variant(force)
            st, y = pl.forward_f32(ctx, x)
            ctx.synchronize()
            got = y.cpu().numpy()
            nan = np.isnan(want)
            assert st == 0 and "k64" in ctx.last_variant, ctx.last_variant
            assert (np.isnan(got) == nan).all() and (got.view(np.uint32)[~nan] == want.view(np.uint32)[~nan]).all(), ctx.last_variant
            seen.add(ctx.last_variant.rsplit(".", 1)[1])
    finally:
        vx.force_variant(None)
        pl.close()
    assert seen == {"t64x64k64", "t64x32k64", "t32x32k64"}, seen


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("k", [100, 256, 300, 512, 641, 1024])
def test_wide_tiles_in_groups_of_256(ctx, oracle, k, bits):
    """One to eight k-blocks, the last group one or two of them: the oracle's bits."""
    import torch
    import volvoxai_amd as vx
    rows, n = 161, 140
    c = cases.packed_case(rows, k, n, 256, k + bits, True)
    w = c["w"] if bits == 8 else cases.four_bit(c["w"])
    words = oracle.pack_w8_words(w) if bits == 8 else oracle.pack_w4_words(w)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, 256, bits=bits)
    pl = vx.PackedLinear(words, c["scales"], c["bias"], k, n, 256, weight_bits=bits)
    x = torch.from_numpy(c["x"]).cuda()
    try:
        for tile in ["t128x128k64"] + ["t128x256k64s3"] * (bits == 8):
            vx.force_variant("a8-mfma." + tile)
            st, y = pl.forward_f32(ctx, x)
            ctx.synchronize()
            assert st == 0 and ctx.last_variant.endswith(tile), ctx.last_variant
            assert (y.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all(), ctx.last_variant
    finally:
        vx.force_variant(None)
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,bits,group,grouped,tile", [
    (333, 256, 14336, 8, 128, True, "t128x128k64"),     # the fold costs both tiles the same
    (333, 256, 14336, 8, 128, False, "t64x64k64"),      # the products fit beside the narrow tile alone
    (874, 4096, 5920, 8, 64, False, "t128x128k64"),
    (874, 4096, 5920, 8, 128, False, "t128x256k64s3"),
    (235, 256, 5120, 4, 128, True, "t32x32k64"),
    (235, 256, 5120, 4, 256, True, "t64x32k64"),
])
def test_the_tile_follows_the_fold(ctx, rows, k, n, bits, group, grouped, tile):
    """The lines of the rule at 256 compute units, where each side was the faster one."""
    import torch
    import volvoxai_amd as vx
    from volvoxai_amd.decoder import pack_w4_words, pack_w8_words
    rng = np.random.default_rng(rows)
    words = (pack_w8_words if bits == 8 else pack_w4_words)(rng.integers(-7, 8, (n, k)).astype(np.int8))
    scales = np.full((n, (k + group - 1) // group), 0.01, np.float32)
    scales[0, 0] += grouped * 0.001
    pl = vx.PackedLinear(words, scales, np.zeros(n, np.float32), k, n, group, weight_bits=bits)
    try:
        st, _ = pl.forward_f32(ctx, torch.ones((rows, k), device="cuda"))
        ctx.synchronize()
        assert st == 0 and ctx.last_variant.endswith(tile), ctx.last_variant
    finally:
        pl.close()
