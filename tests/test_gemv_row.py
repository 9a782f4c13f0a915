"""One and two f32 rows through PackedLinear in one launch (gemv_row.hip) at the edges of its instances."""
import numpy as np
import pytest

import _cases as cases


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("bits,group", [(8, 32), (8, 64), (8, 128), (8, 256), (4, 32), (4, 64), (4, 128), (4, 256)])
@pytest.mark.parametrize("k,n", [(2, 33), (1023, 40), (1024, 2049), (1025, 31), (2050, 64), (3072, 2080), (3101, 8), (4097, 70),
                                 (8192, 33), (8200, 2056), (14336, 24)])
def test_rows_at_the_edges_of_the_instances(ctx, oracle, k, n, bits, group, rows):
    """Lengths on both sides of every instance, both widths of a workgroup's channels (the line is at 64 panels),
    every scale group, n that ends inside a panel: the oracle's bits."""
    import torch
    import volvoxai_amd as vx
    c = cases.packed_case(rows, k, n, group, k + n + bits, True)
    w = c["w"] if bits == 8 else cases.four_bit(c["w"])
    words = oracle.pack_w8_words(w) if bits == 8 else oracle.pack_w4_words(w)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, group, bits=bits)
    pl = vx.PackedLinear(words, c["scales"], c["bias"], k, n, group, weight_bits=bits)
    try:
        for force in (None, "gemv.nofit.row8", "gemv.nofit.row32"):
            vx.force_variant(force)
            st, y = pl.forward_f32(ctx, torch.from_numpy(c["x"]).cuda())
            ctx.synchronize()
            assert st == 0 and ctx.last_variant.endswith("-prep"), ctx.last_variant
            assert (y.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all(), ctx.last_variant
    finally:
        vx.force_variant(None)
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("bits,group", [(8, 32), (8, 256), (4, 32), (4, 128)])
@pytest.mark.parametrize("k,n", [(4608, 40), (6144, 33), (6145, 31), (8193, 64), (10240, 40), (10241, 31), (12288, 33), (12289, 8)])
def test_long_rows_at_the_edges_of_the_instances(ctx, oracle, k, n, bits, group, rows):
    test_rows_at_the_edges_of_the_instances(ctx, oracle, k, n, bits, group, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("no_alloc", [False, True])
@pytest.mark.parametrize("rows,k", [(1, 1024), (2, 10240)])
def test_rows_that_are_overwritten_by_their_output(ctx, oracle, rows, k, no_alloc):
    """In place the workgroups of one launch would read what others have already stored: the rows are prepared first."""
    import torch
    import volvoxai_amd as vx
    c = cases.packed_case(rows, k, k, 128, k, True)
    words = oracle.pack_w8_words(c["w"])
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], k, 128)
    pl = vx.PackedLinear(words, c["scales"], c["bias"], k, k, 128)
    try:
        x = torch.from_numpy(c["x"]).cuda()
        st, _ = pl.forward_f32(ctx, x, out=x, no_alloc=no_alloc)
        ctx.synchronize()
        assert st == 0 and not ctx.last_variant.endswith("-prep"), ctx.last_variant
        assert (x.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
    finally:
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("bits,group", [(8, 32), (8, 128), (4, 32), (4, 128)])
@pytest.mark.parametrize("k,n", [(1, 40), (2, 2100), (8193, 2080), (12001, 70), (14336, 2049)])
def test_fused_swiglu_rows_at_the_ends_of_their_lengths(ctx, oracle, k, n, bits, group, rows):
    """From a single element to the longest row, gate and up both held: the bits of the separate launches."""
    import torch
    import volvoxai_amd as vx
    from volvoxai_amd.w8a8 import swiglu_prepare_i8
    c = cases.packed_case(rows, k, n, group, k + n + bits, True)
    w = c["w"] if bits == 8 else cases.four_bit(c["w"])
    words = oracle.pack_w8_words(w) if bits == 8 else oracle.pack_w4_words(w)
    pl = vx.PackedLinear(words, c["scales"], c["bias"], k, n, group, weight_bits=bits)
    rng = np.random.default_rng(k)
    x = torch.from_numpy(rng.normal(0, 2, (rows, 2 * k)).astype(np.float32)).cuda()
    resid = torch.from_numpy(rng.normal(0, 1, (rows, n)).astype(np.float32)).cuda()
    try:
        st, y = pl.forward_a8(ctx, *swiglu_prepare_i8(ctx, x))
        want = resid + y
        handled, got = pl.forward_fused(ctx, x, vx.ROW_OP_SWIGLU, add_to=resid)
        ctx.synchronize()
        assert st == 0 and handled == 1 and "-swiglu" in ctx.last_variant, ctx.last_variant
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)), ctx.last_variant
    finally:
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,bits,group,route", [
    (1, 8193, 4096, 8, 128, "row8-prep"), (1, 8193, 4097, 8, 128, "row32-prep"), (2, 8193, 4096, 8, 128, "row32-prep"),
    (1, 8192, 4096, 8, 128, "row32-prep"), (1, 4097, 4096, 4, 32, "row8-prep"), (1, 4097, 4096, 4, 64, "row32-prep"),
])
def test_channels_of_a_workgroup(ctx, oracle, rows, k, n, bits, group, route):
    """One long row goes on with eight channels a workgroup to N = 4096 (256 compute units): the oracle's bits there."""
    import torch
    import volvoxai_amd as vx
    c = cases.packed_case(rows, k, n, group, k + n, True)
    w = c["w"] if bits == 8 else cases.four_bit(c["w"])
    words = oracle.pack_w8_words(w) if bits == 8 else oracle.pack_w4_words(w)
    _, want = oracle.packed_linear(c["x"], words, c["scales"], c["bias"], n, group, bits=bits)
    pl = vx.PackedLinear(words, c["scales"], c["bias"], k, n, group, weight_bits=bits)
    try:
        st, y = pl.forward_f32(ctx, torch.from_numpy(c["x"]).cuda())
        ctx.synchronize()
        assert st == 0 and ctx.last_variant.endswith(route), ctx.last_variant
        assert (y.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
    finally:
        pl.close()
