"""QLinear tiles with K split over a workgroup's wavefronts (qlinear_split.hip): edges of tiles and k-blocks, every form of the call, and the
calls that take them."""
import numpy as np
import pytest

import _cases as cases


@pytest.mark.gpu
@pytest.mark.parametrize("zero_points", [False, True])
@pytest.mark.parametrize("unsigned", [False, True])
@pytest.mark.parametrize("rows,k,n", [(33, 1, 1), (40, 16, 4), (32, 127, 31), (47, 128, 32), (64, 129, 33), (65, 512, 34), (17, 513, 36),
                                      (100, 1001, 70), (96, 1024, 130), (33, 4096, 48), (1, 300, 40)])
def test_bytes_at_the_edges(ctx, oracle, rows, k, n, unsigned, zero_points):
    """One k-block to more than eight (some wavefronts without one, a last round of one), rows, channels and columns that end inside a tile,
    both activation types, weight zero points: the oracle's bytes, accumulators and dequantized values."""
    import torch
    import volvoxai_amd as vx
    rng = np.random.default_rng(rows * 7 + k + n)
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    zps = rng.integers(-9, 10, n).astype(np.int32) * int(zero_points)
    scales, bias = rng.uniform(0.005, 0.02, n).astype(np.float32), rng.integers(-2000, 2001, n).astype(np.int32)
    lo, kind, dtype, zp_in = (0, np.uint8, vx.DTYPE_U8, 121) if unsigned else (-128, np.int8, vx.DTYPE_I8, -3)
    x = rng.integers(lo, lo + 256, (rows, k)).astype(kind)
    s_out = float(0.02 * 0.0125 * 74 * 74 * np.sqrt(k) / 40)
    ok, want, want_acc = oracle.qlinear(x, w, bias, scales, zps, 0.02, zp_in, s_out, 5, dtype, vx.DTYPE_I8, vx.DTYPE_I8, want_acc=True)
    assert ok == 1
    lin = vx.QLinear(w, scales, zps, bias, vx.DTYPE_I8)
    try:
        vx.force_variant("mfma-i8.t32x32split")
        ok, y, acc = lin.forward(ctx, torch.from_numpy(x).cuda(), 0.02, zp_in, s_out, 5, input_dtype=dtype, want_accumulators=True)
        ctx.synchronize()
        assert ok == 1 and ctx.last_variant.endswith("t32x32split"), ctx.last_variant
        assert (y.cpu().numpy() == want).all() and (acc.cpu().numpy() == want_acc).all()
    finally:
        vx.force_variant(None)
        lin.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n", [(33, 300, 40), (64, 1024, 33), (70, 2049, 129)])
def test_per_row_scales(ctx, oracle, rows, k, n):
    import torch
    import volvoxai_amd as vx
    c = cases.rowscale_case(rows, k, n, rows + k)
    _, want, _ = oracle.qlinear_rowscale(c["x"], c["w"], c["scales"], c["zps"], c["row_scales"], c["s_out"], 0, bias_f32=c["bias_f32"])
    lin = vx.QLinear(c["w"], c["scales"], c["zps"], None, vx.DTYPE_I8)
    try:
        vx.force_variant("mfma-i8-rowscale.t32x32split")
        ok, y = lin.forward_rowscale(ctx, torch.from_numpy(c["x"]).cuda(), torch.from_numpy(c["row_scales"]).cuda(), c["s_out"], 0,
                                     bias_f32=torch.from_numpy(c["bias_f32"]).cuda())
        ctx.synchronize()
        assert ok == 1 and ctx.last_variant.endswith("t32x32split"), ctx.last_variant
        assert (y.cpu().numpy() == want).all()
    finally:
        vx.force_variant(None)
        lin.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,taken", [(16, 4096, 512, False), (17, 4096, 512, True), (17, 2047, 512, False), (32, 2048, 8192, True),
                                            (32, 2048, 8224, False), (256, 512, 1024, True), (288, 512, 1024, False), (256, 1536, 1536, True),
                                            (288, 1536, 1536, False), (128, 2560, 4096, True), (160, 2560, 4096, False)])
def test_which_calls_take_it(ctx, rows, k, n, taken):
    """The lines of the rule at 256 compute units; signed, unsigned and f32 rows (quantized in front, dequantized behind) the same bytes as the
    kernel that took the call before."""
    import torch
    import volvoxai_amd as vx
    rng = np.random.default_rng(rows)
    lin = vx.QLinear(rng.integers(-127, 128, (n, k)).astype(np.int8), rng.uniform(0.005, 0.02, n).astype(np.float32), np.zeros(n, np.int32),
                     rng.integers(-2000, 2001, n).astype(np.int32), vx.DTYPE_I8)
    f32 = torch.from_numpy(rng.normal(0, 0.6, (rows, k)).astype(np.float32)).cuda()
    s_out = float(0.02 * 0.0125 * 30 * 74 * np.sqrt(k) / 40)

    def outputs():
        outs = []
        for zp, kind, dtype in ((0, torch.int8, vx.DTYPE_I8), (121, torch.uint8, vx.DTYPE_U8)):
            q = (f32 / 0.02 + zp).round().clamp(-127 if zp == 0 else 0, 127 if zp == 0 else 255).to(kind)
            ok, y = lin.forward(ctx, q, 0.02, zp, s_out, 0, input_dtype=dtype)
            assert ok == 1
            outs.append((y, ctx.last_variant))
        ok, y, _ = lin.forward_f32(ctx, f32, 0.02, 0, s_out, 0, input_dtype=vx.DTYPE_I8)
        assert ok == 1
        return outs + [(y, ctx.last_variant)]

    try:
        mine = outputs()
        vx.force_variant("mfma-i8.t64x64")
        before = outputs()
        vx.force_variant(None)
        ctx.synchronize()
        assert ("t32x32split" in mine[0][1]) == taken, mine[0][1]
        for (got, route), (want, _) in zip(mine, before):
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), route
    finally:
        vx.force_variant(None)
        lin.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,n,taken", [(70, 256, 512, False), (70, 257, 512, True), (67, 200, 256, False), (52, 256, 3840, True)])
def test_two_k_blocks(ctx, rows, k, n, taken):
    """Few tiles of up to two k-blocks stay with the tiles of 64 x 64."""
    test_which_calls_take_it(ctx, rows, k, n, taken)


@pytest.mark.gpu
@pytest.mark.parametrize("unsigned", [False, True])
@pytest.mark.parametrize("zero_points", [False, True])
@pytest.mark.parametrize("rows,k,n,taken", [(17, 4096, 512, True), (32, 2048, 2048, True), (24, 2056, 100, True), (16, 4096, 512, False),
                                            (17, 2032, 512, False), (33, 512, 64, True)])
def test_both_activation_types_take_it(ctx, oracle, rows, k, n, taken, zero_points, unsigned):
    """Signed and unsigned bytes of the same extents run on the same kernels, where the rows are read in place and where they are staged:
    the oracle's bytes."""
    import torch
    import volvoxai_amd as vx
    rng = np.random.default_rng(rows + k)
    w, zps = rng.integers(-127, 128, (n, k)).astype(np.int8), rng.integers(-9, 10, n).astype(np.int32) * int(zero_points)
    scales, bias = rng.uniform(0.005, 0.02, n).astype(np.float32), rng.integers(-2000, 2001, n).astype(np.int32)
    lo, kind, dtype, zp_in = (0, np.uint8, vx.DTYPE_U8, 121) if unsigned else (-128, np.int8, vx.DTYPE_I8, -3)
    x = rng.integers(lo, lo + 256, (rows, k)).astype(kind)
    s_out = float(0.02 * 0.0125 * 74 * 74 * np.sqrt(k) / 40)
    ok, want = oracle.qlinear(x, w, bias, scales, zps, 0.02, zp_in, s_out, 5, dtype, vx.DTYPE_I8, vx.DTYPE_I8)
    assert ok == 1
    lin = vx.QLinear(w, scales, zps, bias, vx.DTYPE_I8)
    try:
        ok, y = lin.forward(ctx, torch.from_numpy(x).cuda(), 0.02, zp_in, s_out, 5, input_dtype=dtype)
        ctx.synchronize()
        assert ok == 1 and ("t32x32split" in ctx.last_variant) == taken, ctx.last_variant
        assert (y.cpu().numpy() == want).all()
    finally:
        lin.close()
