"""The dequantizing linear with K split over a workgroup's wavefronts (linear_slabs.hip) at the edges of its slabs, passes and tiles,
and the calls that take it."""
import numpy as np
import pytest

import _cases as cases


def _linear(oracle, k, n, group, bits, c):
    import volvoxai_amd as vx
    w = c["w"] if bits == 8 else cases.four_bit(c["w"])
    words = oracle.pack_w8_words(w) if bits == 8 else oracle.pack_w4_words(w)
    return words, vx.PackedLinear(words, c["scales"], c["bias"], k, n, group, weight_bits=bits)


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("rows,k,n", [(1, 1, 1), (16, 32, 16), (17, 33, 17), (32, 128, 32), (33, 129, 33), (31, 300, 47), (5, 1023, 63),
                                      (47, 1025, 64), (64, 2048, 65), (65, 2079, 257), (70, 2500, 300)])
def test_tiles_at_their_edges(ctx, oracle, rows, k, n, group, bits):
    """One column to more than two passes of every group size, last passes of one wavefront and of all, an odd group in the last slab of
    two and half a group of 256, rows and channels that end inside a tile, rows that are not finite: the oracle's bits on every tile."""
    import torch
    import volvoxai_amd as vx
    c = cases.packed_case(rows, k, n, group, rows + k + n + bits, True, special_rows=rows == 47)
    words, pl = _linear(oracle, k, n, group, bits, c)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, group, bits=bits)
    nan = np.isnan(want)
    x = torch.from_numpy(c["x"]).cuda()
    try:
        for tile in ("slab16x16", "slab16x32", "slab32x32"):
            vx.force_variant("a8-mfma." + tile)
            st, y = pl.forward_f32(ctx, x, out=torch.full((rows, n), 7.0, device="cuda"))
            ctx.synchronize()
            got = y.cpu().numpy()
            # (up to two rows, and a few more short ones, go in one launch whatever tile is named)
            assert st == 0 and (ctx.last_variant.endswith(tile) or rows <= 2), ctx.last_variant
            assert (np.isnan(got) == nan).all() and (got.view(np.uint32)[~nan] == want.view(np.uint32)[~nan]).all(), ctx.last_variant
    finally:
        vx.force_variant(None)
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,bits,group,tile", [
    (64, 4096, 512, 8, 128, "slab16x16"), (64, 4096, 4096, 8, 128, "slab32x32"), (32, 4096, 4096, 8, 128, "slab16x32"),
    (128, 4096, 4096, 8, 128, None), (257, 4096, 64, 8, 128, None), (96, 1279, 64, 8, 128, None), (96, 1280, 64, 8, 128, "slab16x16"),
    (8, 4096, 64, 8, 128, None), (8, 2500, 64, 8, 128, "slab16x16"), (4, 4096, 64, 8, 128, None), (4, 4097, 64, 8, 128, "slab16x16"),
    (16, 2000, 8000, 4, 128, "slab16x16"), (24, 4096, 14336, 8, 128, None), (24, 4000, 8192, 8, 128, None), (16, 2048, 14336, 8, 64, None), (16, 4096, 6144, 8, 64, "slab16x16")])
def test_which_calls_take_it(ctx, rows, k, n, bits, group, tile):
    """The lines of the rule at 256 compute units; both entry points agree bit for bit, and with the kernel that took the call before."""
    import torch
    import volvoxai_amd as vx
    from volvoxai_amd.decoder import pack_w4_words, pack_w8_words
    rng = np.random.default_rng(rows)
    words = (pack_w8_words if bits == 8 else pack_w4_words)(rng.integers(-7, 8, (n, k)).astype(np.int8))
    scales = rng.uniform(0.002, 0.01, (n, (k + group - 1) // group)).astype(np.float32)
    pl = vx.PackedLinear(words, scales, rng.normal(0, 0.1, n).astype(np.float32), k, n, group, weight_bits=bits)
    x = torch.from_numpy(rng.normal(0, 1, (rows, k)).astype(np.float32)).cuda()
    try:
        st, y = pl.forward_f32(ctx, x)
        assert st == 0 and ("slab" in ctx.last_variant) == bool(tile) and (not tile or ctx.last_variant.endswith(tile)), ctx.last_variant
        st, again = pl.forward_f32(ctx, x, out=torch.empty_like(y), no_alloc=True)
        assert st == 0 and ("slab" in ctx.last_variant) == bool(tile), ctx.last_variant
        vx.force_variant("a8-mfma.t64x64k64")
        st, plain = pl.forward_f32(ctx, x)
        vx.force_variant(None)
        ctx.synchronize()
        assert st == 0 and torch.equal(y.view(torch.int32), again.view(torch.int32)) and torch.equal(y.view(torch.int32), plain.view(torch.int32))
    finally:
        vx.force_variant(None)
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,bits,group,tile", [
    (24, 8192, 8192, 8, 128, "slab32x32"), (16, 14336, 8192, 8, 128, "slab16x16"),  # no instance: its LDS does not suffice
    (6, 3000, 1531, 8, 64, "slab16x16"), (8, 3000, 7000, 8, 64, "slab16x16"),       # none: the last group is half a group
    (8, 14336, 8192, 8, 128, "slab16x16"), (8, 8192, 8192, 4, 128, "slab16x16"),    # one that reads its rows from memory
    (8, 4096, 14336, 8, 64, "slab16x16"), (16, 8192, 14336, 8, 128, "slab16x16"),
    (4, 8192, 14336, 8, 128, None), (8, 4096, 8192, 8, 128, None),                  # one that has them in LDS
    (10, 6000, 8192, 8, 128, None), (3, 10000, 5055, 8, 128, None), (24, 6000, 5055, 8, 128, None), (8, 13000, 4096, 8, 128, "slab16x16"),
    (8, 10000, 8192, 4, 256, None), (8, 6000, 8192, 4, 128, "slab16x16"), (24, 10000, 5055, 8, 128, "slab16x32"),   # the general kernel, and not
    (239, 2304, 736, 8, 256, None), (112, 2304, 736, 8, 256, "slab16x16"), (118, 1536, 1280, 8, 128, None), (118, 1536, 1024, 8, 128, "slab16x32")])  # cheap folds
def test_what_stands_behind_a_call(ctx, rows, k, n, bits, group, tile):
    """What the rule takes to stand behind a call is what the streaming kernel's launcher has for it; short walks and cheap folds are left to
    the tiles of gemm_k64.hip."""
    test_which_calls_take_it(ctx, rows, k, n, bits, group, tile)


@pytest.mark.gpu
def test_scratch_with_room_for_the_rows_alone(oracle):
    """225 rows of 18000 fit the fixed scratch array (4 MiB) and a scratch reserved for them, eight tiles of 32 rows do not: the call is
    taken as before, and by the slab kernel where its scratch may grow."""
    import torch
    import volvoxai_amd as vx
    rows, k, n, group = 225, 18000, 40, 128
    c = cases.packed_case(rows, k, n, group, 5, True)
    words, pl = _linear(oracle, k, n, group, 8, c)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, group)
    x = torch.from_numpy(c["x"]).cuda()
    fixed, reserved, growing = vx.Context(0, None), vx.Context(0, None), vx.Context(0, None)
    try:
        reserved.reserve_scratch(3 << 20)  # (in whole MiB, with one to spare)
        out = torch.empty((rows, n), device="cuda")
        for context, slabs, no_alloc in ((fixed, False, True), (reserved, False, False), (growing, True, False)):
            out.fill_(7.0)
            torch.cuda.synchronize()
            st, _ = pl.forward_f32(context, x, out=out, no_alloc=no_alloc)
            context.synchronize()
            assert st == 0 and ("slab" in context.last_variant) == slabs, context.last_variant
            assert (out.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
    finally:
        pl.close(), fixed.close(), reserved.close(), growing.close()


@pytest.mark.gpu
def test_scratch_grows_for_the_tiles_outside_a_recording(oracle):
    """A context whose scratch, sized by a smaller call, holds 70 rows of 14336 and not three tiles of 32 of them: it grows, unless the
    launches are being recorded, by the context or by the owner of its stream, which is refused nothing it was given before."""
    import torch
    import volvoxai_amd as vx
    rows, k, n, group = 70, 14336, 40, 128
    c = cases.packed_case(rows, k, n, group, 5, True)
    words, pl = _linear(oracle, k, n, group, 8, c)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, group)
    x, out = torch.from_numpy(c["x"]).cuda(), torch.empty((rows, n), device="cuda")

    def context(stream):
        made = vx.Context(0, stream)
        st, _ = pl.forward_f32(made, x[:40].contiguous(), out=torch.empty((40, n), device="cuda"))
        made.synchronize()
        assert st == 0
        return made

    def same():
        torch.cuda.synchronize()
        equal = (out.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
        out.fill_(7.0)
        torch.cuda.synchronize()
        return equal

    stream = torch.cuda.Stream()
    recording, capturing, growing = context(None), context(stream), context(None)
    try:
        recording.begin_recording()
        st, _ = pl.forward_f32(recording, x, out=out)
        replay = recording.end_recording()
        assert st == 0 and "slab" not in recording.last_variant, recording.last_variant
        for _ in range(2):
            replay.launch(recording)
            assert same()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            st, _ = pl.forward_f32(capturing, x, out=out)
        assert st == 0 and "slab" not in capturing.last_variant, capturing.last_variant
        for _ in range(2):
            graph.replay()
            assert same()
        for made in (growing, recording, capturing):
            st, _ = pl.forward_f32(made, x, out=out)
            made.synchronize()
            assert st == 0 and "slab" in made.last_variant and same(), made.last_variant
        replay.launch(recording)  # (its block is kept)
        assert same()
        replay.close()
    finally:
        pl.close(), recording.close(), capturing.close(), growing.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,tile", [(1000, 1531, "t64x32k64"), (640, 4096, "t64x32k64"), (900, 4096, "t64x64k64"), (768, 4096, "t64x64k64")])
def test_tiles_of_groups_of_32(ctx, oracle, rows, n, tile):
    """More 64x64 tiles than 1.5 a compute unit (256 of them): the half tiles where they need an odd number of rounds of the device."""
    import torch
    c = cases.packed_case(rows, 96, n, 32, rows, True)
    words, pl = _linear(oracle, 96, n, 32, 8, c)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, 32)
    try:
        st, y = pl.forward_f32(ctx, torch.from_numpy(c["x"]).cuda())
        ctx.synchronize()
        assert st == 0 and ctx.last_variant.endswith(tile), ctx.last_variant
        assert (y.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
    finally:
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows,n,tile", [(1000, 1531, "t64x32k64"), (720, 4500, "t64x64k64"), (1500, 3000, "t64x64k64"), (2048, 5184, "t64x64k64"), (2048, 13888, "t64x64k64")])
def test_tiles_of_groups_of_32_in_many_rounds(ctx, rows, n, bits, tile):
    """An odd number of rounds of half tiles saves less and less of the launch, and a half tile costs more than half: three against two are
    taken, seven against four and more are not.  The same bits as the other tile."""
    import torch
    import volvoxai_amd as vx
    from volvoxai_amd.decoder import pack_w4_words, pack_w8_words
    rng = np.random.default_rng(n)
    words = (pack_w8_words if bits == 8 else pack_w4_words)(rng.integers(-7, 8, (n, 64)).astype(np.int8))
    pl = vx.PackedLinear(words, rng.uniform(0.002, 0.01, (n, 2)).astype(np.float32), np.zeros(n, np.float32), 64, n, 32, weight_bits=bits)
    x = torch.from_numpy(rng.normal(0, 1, (rows, 64)).astype(np.float32)).cuda()
    try:
        st, y = pl.forward_f32(ctx, x)
        assert st == 0 and ctx.last_variant.endswith(tile), ctx.last_variant
        vx.force_variant("a8-mfma." + {"t64x32k64": "t64x64k64", "t64x64k64": "t64x32k64"}[tile])
        st, other = pl.forward_f32(ctx, x)
        ctx.synchronize()
        assert st == 0 and not ctx.last_variant.endswith(tile) and torch.equal(y.view(torch.int32), other.view(torch.int32))
    finally:
        vx.force_variant(None)
        pl.close()
