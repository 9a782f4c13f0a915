"""The C-ABI library loads without a GPU, exports every declared symbol, and
fails loudly (never silently on a CPU path) when there is no device."""
import ctypes as C
import re
from pathlib import Path

import numpy as np
import pytest

import volvoxai_amd as vx
from volvoxai_amd._lib import declared_symbols, library

ROOT = Path(__file__).resolve().parent.parent


def test_library_exports_every_declared_symbol():
    lib = library()
    names = declared_symbols()
    assert len(names) >= 30
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in include/vxhip_w8a8.h but not exported"
    assert lib.vxhip_abi_version() == 1


def test_kernel_variant_table_shape():
    rows = vx.kernel_variants()
    ids = {r["id"] for r in rows}
    assert {"hip.qlinear.mfma-i8", "hip.qlinear.gemv-mfma", "hip.packed-linear.a8-mfma",
            "hip.packed-linear.a8-gemv-mfma", "hip.packed-linear.w4a8-mfma",
            "hip.packed-linear.w4a8-gemv-mfma"} <= ids
    for r in rows:
        assert r["backend"] == 0 and r["id"].startswith("hip.") and r["priority"] > 0
        assert r["operator_kind"] in (1002, 1005, 1007, 1036)
    # QLinear, QGemm and QMatMul share one kernel family, as upstream's cuda.qlinear.* rows do
    for fam in ("hip.qlinear.mfma-i8", "hip.qlinear.gemv-mfma"):
        assert {r["operator_kind"] for r in rows if r["id"] == fam} == {1002, 1005, 1007}


def test_kernel_variant_table_names_every_linear_kernel():
    """The kernels behind a family's routes, and the matrix instructions they are made of, as the sources have them."""
    rows = vx.kernel_variants()
    sources = [p.read_text() for p in sorted((ROOT / "volvoxai_amd" / "csrc").glob("gem*.hip"))]
    names = {n for text in sources for n in re.findall(r"void (gem[mv]_\w*kernel)\(", text)}
    assert len(names) == 8
    assert names == {e.split("<")[0] for r in rows for e in r["entrypoint_id"].split("|") if e.startswith("gem")}
    used = {n for text in sources for n in re.findall(r"__builtin_amdgcn_mfma_i32_(\w+)_i8\(", text)}
    assert used == {n for r in rows for n in re.findall(r"mfma-i32-(\w+)-i8", r["required_features"])}
    few = [r for r in rows if "gemv_few_kernel" in r["entrypoint_id"]]
    assert len(few) == 2 and all("mfma-i32-16x16x64-i8" in r["required_features"] for r in few)


def _no_gpu():
    return library().vxhip_device_count() == 0


@pytest.mark.skipif(not _no_gpu(), reason="checks the no-device behaviour")
def test_without_device_entry_points_decline_and_say_why():
    lib = library()
    h = C.c_void_p()
    assert lib.vxhip_context_create(0, None, 0, C.byref(h)) == -6  # BACKEND_UNAVAILABLE
    assert not h and b"device" in lib.vxhip_last_error()
    x = np.zeros((2, 16), np.int8)
    w = np.zeros((4, 16), np.int8)
    ok, _ = vx.qlinear_i8u8(x, w, np.ones(4, np.float32), np.zeros(4, np.int32), np.zeros(4, np.int32),
                            2, 16, 4, 1.0, 0, 1.0, 0, vx.DTYPE_I8, vx.DTYPE_I8, vx.DTYPE_I8)
    assert ok == 0  # declined, not computed somewhere else
    st, _ = vx.packed_linear_f32(np.zeros((1, 32), np.float32), np.zeros((2, 8), np.uint32),
                                 np.ones((2, 1), np.float32), None, 32, 2, 32)
    assert st == -1


def test_argument_validation_happens_before_any_device_work():
    lib = library()
    h = C.c_void_p()
    # non-byte dtype, null tensors: INVALID_ARGUMENT regardless of hardware
    assert lib.vxhip_qlinear_create(None, None, None, None, 4, 4, vx.DTYPE_I8, C.byref(h)) == -1
    w = np.zeros((4, 4), np.int8)
    s = np.ones(4, np.float32)
    z = np.zeros(4, np.int32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    assert lib.vxhip_qlinear_create(p(w), p(s), p(z), None, 4, 4, 18, C.byref(h)) == -1
    bad = np.array([1, 1, 0, 1], np.float32)
    if _no_gpu():
        return
    assert lib.vxhip_qlinear_create(p(w), p(bad), p(z), None, 4, 4, vx.DTYPE_I8, C.byref(h)) == -1
    words = np.zeros((2, 8), np.uint32)
    assert lib.vxhip_packed_linear_create(p(words), p(s), None, 32, 2, 32, 4, C.byref(h)) == -7
    assert lib.vxhip_packed_linear_create(p(words), p(s), None, 32, 2, 48, 8, C.byref(h)) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 3, 8, 17, 32, 33, 64])
def test_routes_lie_in_the_row_domains_of_the_table(ctx, rows):
    """The ids that calls report, against the rows their records declare: few rows on the split and the slab kernels too."""
    import torch
    table = {r["id"]: r["predicate_id"] for r in vx.kernel_variants()}
    rng = np.random.default_rng(rows)
    n = 512

    def admitted():
        family = max((i for i in table if ctx.last_variant.startswith(i + ".")), key=len)
        least, most = re.search(r"rows-g[te](\d+)", table[family]), re.search(r"rows-le(\d+)", table[family])
        if least and rows < int(least.group(1)) + ("rows-gt" in table[family]):
            return False
        return not (most and rows > int(most.group(1)))

    for k in (2500, 4608):
        scales = rng.uniform(0.002, 0.01, (n, (k + 127) // 128)).astype(np.float32)
        q = vx.QLinear(rng.integers(-127, 128, (n, k)).astype(np.int8), scales[:, 0].copy(), np.zeros(n, np.int32), np.zeros(n, np.int32), vx.DTYPE_I8)
        words = np.full((n, (k + 3) // 4), 0x81818181, np.uint32)
        p = vx.PackedLinear(words, scales, None, k, n, 128)
        x = torch.ones((rows, k), device="cuda")
        try:
            ok, _ = q.forward(ctx, x.to(torch.int8), 0.02, 0, 1.0, 0, input_dtype=vx.DTYPE_I8)
            assert ok == 1 and admitted(), ctx.last_variant
            st, _ = p.forward_f32(ctx, x)
            assert st == 0 and admitted(), ctx.last_variant
        finally:
            ctx.synchronize()
            q.close(), p.close()
