"""Three to eight f32 rows of PackedLinear in one launch (gemv_few.hip): the oracle's bits at the edges of its instances and
rows, every channel count, every group size and weight width, rows that are not finite, and the lines of its rule."""
import numpy as np
import pytest


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _linear(vx, oracle, rng, k, n, bits, group):
    top = 2 ** (bits - 1) - 1
    w = rng.integers(-top - 1, top + 1, (n, k)).astype(np.int8)
    words = (oracle.pack_w8_words if bits == 8 else oracle.pack_w4_words)(w)
    scales = rng.uniform(0.002, 0.01, (n, (k + group - 1) // group)).astype(np.float32)
    bias = rng.normal(0, 0.1, n).astype(np.float32)
    return vx.PackedLinear(words, scales, bias, k, n, group, weight_bits=bits), words, scales, bias


@pytest.mark.gpu
@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows,k", [(3, 2), (4, 31), (3, 1023), (4, 1025), (3, 2050), (4, 3073), (4, 4096), (5, 33), (8, 1024), (6, 1027),
                                    (7, 2048)])
def test_few_rows_at_their_edges(ctx, oracle, rows, k, bits, group):
    import volvoxai_amd as vx
    rng = np.random.default_rng(rows * k + bits + group)
    for n in (1, 47, 100):
        pl, words, scales, bias = _linear(vx, oracle, rng, k, n, bits, group)
        x = (rng.normal(0, 1, (rows, k)) * rng.uniform(1e-3, 50, (rows, 1))).astype(np.float32)
        x[1] = 0.0
        x[rows - 1, k - 1] = np.inf
        x[0, 0] *= 300.0
        want = oracle.packed_linear(x, words, scales, bias, n, group, bits=bits)[1]
        # what the rule takes is built: 64 channels a workgroup for up to four rows and eight bits in groups of 64 and more,
        # 32 for up to four rows, and for more of up to 1024
        wide = 16 if rows > 4 and k > 1024 else 32
        widest = 64 if rows <= 4 and bits == 8 and group > 32 else wide
        for force, ch in (("gemv.few16", 16), ("gemv.few32", wide), ("gemv.few64", widest), (None, 16)):
            vx.force_variant(force)
            st, y = pl.forward_f32(ctx, _dev(x))
            ctx.synchronize()
            vx.force_variant(None)
            got = y.cpu().numpy()
            assert st == 0 and ctx.last_variant.endswith(f".few{ch}"), ctx.last_variant
            nan = np.isnan(want)
            assert (np.isnan(got) == nan).all() and (got.view(np.uint32)[~nan] == want.view(np.uint32)[~nan]).all(), ctx.last_variant
        pl.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,few", [(3, 4096, 14336, "few64"), (4, 4096, 4096, "few16"), (4, 4097, 512, None), (5, 1024, 8192, "few32"),
                                          (8, 1024, 8193, None), (8, 2048, 4096, "few16"), (5, 2048, 4097, None), (8, 2049, 64, None),
                                          (9, 512, 64, None), (3, 1, 64, None)])
def test_the_rule_and_the_prepared_rows_give_the_same_bits(ctx, oracle, rows, k, n, few):
    """On both sides of the rule's lines, against the preparation and the linear as launches of their own; and an output
    that overlaps its input goes by way of the prepared rows."""
    import torch
    import volvoxai_amd as vx
    rng = np.random.default_rng(k + n)
    pl, *_ = _linear(vx, oracle, rng, k, n, 8, 128)
    x = _dev(rng.normal(0, 1, (rows, k)).astype(np.float32))
    a8, sc = vx.w8a8.packed_prepare_i8(ctx, x)
    st0, want = pl.forward_a8(ctx, a8, sc)
    st1, y = pl.forward_f32(ctx, x)
    ctx.synchronize()
    assert st0 == st1 == 0 and ctx.last_variant.endswith(few if few else "") and (".few" in ctx.last_variant) == bool(few), ctx.last_variant
    assert torch.equal(y.view(torch.int32), want.view(torch.int32))
    if n <= k:
        buf = torch.zeros(rows * k, device="cuda")
        buf[:] = x.reshape(-1)
        st2, _ = pl.forward_f32(ctx, buf.view(rows, k), out=buf[:rows * n].view(rows, n))
        ctx.synchronize()
        assert st2 == 0 and ".few" not in ctx.last_variant
        assert torch.equal(buf[:rows * n].view(rows, n).view(torch.int32), want.view(torch.int32))
    pl.close()
