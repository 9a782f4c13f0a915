"""The row kernels (row_prepare.hip) at the edges of their instances: rows that end inside a 16-byte piece or a
16-byte chunk of codes, lengths on both sides of every thread and pass count, few and many rows, both layouts."""
import numpy as np
import pytest


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [2, 32, 257])
@pytest.mark.parametrize("d", [1, 6, 18, 1021, 1024, 1025, 2049, 3075, 4096, 4100, 8192, 8195, 14340])
@pytest.mark.parametrize("op", ["plain", "norm", "swiglu"])
def test_row_kernels_at_their_edges(oracle, op, d, rows):
    """Codes and scales are exactly the oracle's preparation of the kernel's f32 rows; those rows follow the
    double-precision definition to one rounding (RMSNorm) and to the f32 steps of SwiGLU (three roundings of
    2^-24 and the exponential's two units: below 5 * 2^-23)."""
    import torch
    import volvoxai_amd as vxa
    import volvoxai_amd.w8a8 as vx
    if rows == 257 and d not in (18, 1025, 3075, 8195, 14340):
        pytest.skip("many rows: one length per instance")
    rng = np.random.default_rng(d * 3 + rows)
    width = 2 * d if op == "swiglu" else d
    x = (rng.normal(0, 1, (rows, width)) * rng.uniform(0.1, 8, (rows, 1))).astype(np.float32)
    x[1, width // 2] = np.inf if d > 1 else x[1, 0]
    gain = rng.uniform(0.5, 1.5, d).astype(np.float32)
    got = {}
    for operand in (False, True):
        ctx = vxa.Context(0, torch.cuda.current_stream())
        ctx.set_activation_layout(operand)
        if op == "norm":
            got[operand] = vx.rmsnorm_prepare_i8(ctx, _dev(x), _dev(gain), 1e-6, want_normalized=True)
        elif op == "swiglu":
            got[operand] = vx.swiglu_prepare_i8(ctx, _dev(x), want_activated=True)
        else:
            got[operand] = (*vx.packed_prepare_i8(ctx, _dev(x)), _dev(x))
        ctx.synchronize()
        got[operand] = [t.cpu().numpy() for t in got[operand]]
        ctx.close()
    codes, scales, values = got[False]
    xd = x.astype(np.float64)
    with np.errstate(all="ignore"):
        if op == "norm":
            want = xd * (1.0 / np.sqrt((xd * xd).mean(-1, keepdims=True) + 1e-6)) * gain.astype(np.float64)
            bound = 2.0 ** -23
        elif op == "swiglu":
            want = xd[:, :d] / (1.0 + np.exp(-xd[:, :d])) * xd[:, d:]
            bound = 5 * 2.0 ** -23
        else:
            want, bound = xd, 0.0
    finite = np.isfinite(want).all(-1)
    assert (np.abs(values[finite] - want[finite]) <= bound * np.abs(want[finite])).all()
    want_codes, want_scales, fin = oracle.packed_prepare(values)
    good = fin == 1
    assert (good == finite).all() and (np.isnan(scales) == ~good).all() and not codes[~good].any()
    assert (codes[good] == want_codes[good]).all()
    assert (scales[good].view(np.uint32) == want_scales[good].view(np.uint32)).all()
    if rows <= 32:
        bcodes, bscales, _ = got[True]
        by_chunk = bcodes.reshape(-1, 32, 16)[:, :rows].transpose(1, 0, 2).reshape(rows, -1)
        assert (by_chunk[:, :d] == codes).all() and not by_chunk[:, d:].any()
        assert (bscales.view(np.uint32) == scales.view(np.uint32)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["plain", "norm", "swiglu"])
@pytest.mark.parametrize("d", [5121, 6144, 6146, 8196, 10240, 10243, 12288, 12291])
def test_many_long_rows(oracle, op, d):
    """More rows than compute units, lengths on both sides of every number of passes."""
    test_row_kernels_at_their_edges(oracle, op, d, 259)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,d", [(3, 1022), (32, 2048), (300, 4099)])
def test_residual_add_rides_in_front_of_the_norm(ctx, rows, d):
    import torch
    import volvoxai_amd.w8a8 as vx
    rng = np.random.default_rng(d)
    x, delta = (_dev(rng.normal(0, 1, (rows, d)).astype(np.float32)) for _ in range(2))
    gain = _dev(rng.uniform(0.5, 1.5, d).astype(np.float32))
    total = x + delta
    want_codes, want_scales = vx.rmsnorm_prepare_i8(ctx, total, gain, 1e-5)
    codes, scales = vx.add_rmsnorm_prepare_i8(ctx, x, delta, gain, 1e-5)
    ctx.synchronize()
    assert torch.equal(x, total) and torch.equal(codes, want_codes) and torch.equal(scales, want_scales)
