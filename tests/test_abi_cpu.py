"""Host-side checks that need no GPU: the C-ABI library loads, exports every symbol that
include/dlt.h declares, and rejects bad arguments before launching anything."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _lib():
    from dl_templates_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("libdlt_hip.so not built (run __graft_entry__.build())")
    return _lib


def test_library_exports_every_declared_symbol():
    L = _lib()
    lib = L.load()
    header = open(os.path.join(ROOT, "include", "dlt.h")).read()
    declared = set(re.findall(r"\b(dlt_[a-z0-9_]+)\s*\(", header))
    declared -= {"dlt_dtype_t"}
    assert declared, "no declarations found in include/dlt.h"
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} is declared in dlt.h but not exported"
    assert set(L.EXPORTS) == declared
    assert lib.dlt_version() >= 1


def test_argument_validation_happens_before_any_launch():
    L = _lib()
    lib = L.load()
    shape = L.SwaShape(1, 1, 1, 4, 4, 1, 1, 64, 64, 1.0, 7)  # bad dtype
    st4 = (ctypes.c_int64 * 4)(1, 1, 1, 1)
    st3 = (ctypes.c_int64 * 3)(1, 1, 1)
    one = ctypes.c_void_p(16)
    rc = lib.dlt_swa_fwd(one, st4, one, st4, one, st4, one, st4, one, st3, shape, None, None)
    assert rc == 1 and b"dtype" in lib.dlt_last_error()
    shape = L.SwaShape(1, 1, 1, 4, 4, 1, 1, 64, 64, 1.0, 0)
    rc = lib.dlt_swa_fwd(None, st4, one, st4, one, st4, one, st4, one, st3, shape, None, None)
    assert rc == 1 and b"NULL" in lib.dlt_last_error()
    shape = L.SwaShape(1, 1, 1, 4, 4, 1, 1, 512, 64, 1.0, 0)
    rc = lib.dlt_swa_fwd(one, st4, one, st4, one, st4, one, st4, one, st3, shape, None, None)
    assert rc == 2 and b"head dims" in lib.dlt_last_error()
    shape = L.SwaShape(1, 1, 1, 4, 4, 1, 1, 64, 64, float("inf"), 0)
    rc = lib.dlt_swa_fwd(one, st4, one, st4, one, st4, one, st4, one, st3, shape, None, None)
    assert rc == 1 and b"sm_scale" in lib.dlt_last_error()
    rc = lib.dlt_flash_fwd(one, st4, one, st4, one, st4, one, st4, one, st3, L.FlashShape(1, 1, 8, 8, 64, 64, float("nan"), 0, 0), None)
    assert rc == 1 and b"sm_scale" in lib.dlt_last_error()
    st5 = (ctypes.c_int64 * 5)(1, 1, 1, 1, 1)
    shape = L.SwaShape(1, 1, 6, 4, 4, 1, 1, 64, 64, 1.0, 0)  # tile of 2 x 2 pixels is not 6 tokens
    rc = lib.dlt_swa_fwd_image(one, st5, one, st5, one, st5, one, st5, one, st3, shape, L.SwaTile(2, 2), None, None)
    assert rc == 1 and b"b_size" in lib.dlt_last_error()
    rc = lib.dlt_swa_image_offsets(0, 4, 2, 2, 8, 1, one, None)
    assert rc == 1 and b"grid" in lib.dlt_last_error()
    fshape = L.FlashShape(1, 1, 8, 16, 64, 64, 1.0, 1, 0)  # causal with Lq != Lk
    rc = lib.dlt_flash_fwd(one, st4, one, st4, one, st4, one, st4, one, st3, fshape, None)
    assert rc == 1 and b"causal" in lib.dlt_last_error()
    rope = L.RopeDesc(16, 16, 16, 16, 16, 8, 4, 4)
    rc = lib.dlt_rope2d(one, st3, 1, 4, 16, rope, 0, 0, None)  # 4R = 32 > C = 16
    assert rc == 1 and b"n_rdim" in lib.dlt_last_error()
    assert lib.dlt_rope2d(None, st3, 0, 0, 16, L.RopeDesc(0, 0, 0, 0, 0, 0, 0, 0), 0, 0, None) == 0


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "dl_templates_amd")
    for fn in os.listdir(pkg):
        if fn.endswith(".py"):
            src = open(os.path.join(pkg, fn)).read()
            assert "oracle" not in src, f"{fn} must not reference the oracle"


def test_table_context_matches_oracle_tables():
    import torch
    from dl_templates_amd.rope2d import FusedRotaryPositionEncodingContext as Ctx
    from dl_templates_amd.fused_rope2d import FusedInplaceRotaryPositionEncoding2D as M
    from oracle import attn_oracle as orc
    assert (Ctx(16, 64).cs_components - orc.rope_tables(8, 64)).abs().max().item() <= 1.2e-7
    assert torch.equal(M.encode_idx(5, 7), orc.encode_idx(5, 7))
    m = M(32, 8, 9)
    assert m.row_buffer.cs_components.shape == (8, 8, 2) and m.col_buffer.cs_components.shape == (9, 8, 2)


def test_rope_operands_on_the_host_raise_before_any_launch():
    """idx / tables are dereferenced by the kernels: the attention wrappers must refuse host tensors (what
    encode_idx returns without a default device) instead of handing a host pointer to the GPU."""
    import pytest
    import torch
    from dl_templates_amd import _lib
    from dl_templates_amd.fused_rope2d import FusedInplaceRotaryPositionEncoding2D as M

    class OnGpu:   # stands in for the CUDA tensor the rotation is applied to (no GPU in the CPU suite)
        is_cuda = True
        device = torch.device("cuda:0")

    idx = M.encode_idx(4, 4)
    tab = torch.zeros(4, 8, 2)
    with pytest.raises(RuntimeError, match="ROCm GPU only"):
        _lib.rope_desc(idx, tab, tab, like=OnGpu())
    with pytest.raises(ValueError, match="entries for"):
        _lib.rope_desc(idx, tab, tab, n_tokens=17)
    with pytest.raises(TypeError):
        _lib.rope_desc(idx.long(), tab, tab)


def test_operators_are_autograd_functions():
    """Drop-in contract: the operators are autograd.Function classes with forward and backward of their own."""
    import torch
    from dl_templates_amd.flash_attn import _attention
    from dl_templates_amd.fused_rope2d import RotaryPE2D
    from dl_templates_amd.tiled_swa import TiledSwa, TiledSwaImage, TiledSwaRope
    for op in (TiledSwa, TiledSwaRope, TiledSwaImage, RotaryPE2D, _attention):
        assert issubclass(op, torch.autograd.Function)
        assert "forward" in vars(op) and "backward" in vars(op)


def test_flash_workspace_of_a_shape():
    L = _lib()
    lib = L.load()

    def need(backward, *shape):
        n = ctypes.c_int64(-1)
        assert lib.dlt_flash_workspace(L.FlashShape(*shape), backward, ctypes.byref(n)) == 0, lib.dlt_last_error()
        return n.value
    # 64 queries x 4000 keys: 8 shares of a forward pass (64 output dims, maximum and sum) and of dQ (512 keys each but the last); dK and dV of 64 keys the same way
    assert need(0, 1, 2, 64, 4000, 64, 64, 0.1, 0, 0) == 4 * 2 * 8 * 64 * (64 + 2)
    assert need(1, 1, 2, 64, 4000, 64, 64, 0.1, 0, 0) == 4 * 2 * 8 * 64 * 64
    assert need(1, 1, 1, 4000, 64, 64, 64, 0.1, 0, 0) == 4 * 8 * 64 * 128
    # on a full chip one workgroup takes all shares of its own block and needs nothing; partial results never exceed the stated maximum
    assert need(0, 2, 95, 64, 4000, 64, 64, 0.1, 0, 0) == 4 * 190 * 8 * 64 * (64 + 2) and need(0, 2, 96, 64, 4000, 64, 64, 0.1, 0, 0) == 0
    for shape in ((64, 32, 512, 8192, 128, 128), (128, 32, 8192, 1024, 64, 64), (1, 1, 40000, 1000000, 128, 128), (1, 1, 1000000, 40000, 64, 128), (1, 90, 128, 8192, 128, 128),
                  (1, 1, 24000, 400000, 128, 128), (1, 1, 24000, 400000, 64, 128), (1, 180, 64, 8192, 64, 128), (1, 1, 400000, 24000, 128, 128)):
        assert need(0, *shape, 0.1, 0, 0) <= 256 << 20 and need(1, *shape, 0.1, 0, 0) <= 256 << 20
    # nothing is split under a mask, for balanced sides, in fp32, at odd head dims and outside the classes of 64 and 128
    for shape in ((1, 1, 4000, 4000, 64, 64, 0.1, 1, 0), (1, 1, 2048, 2048, 64, 64, 0.1, 0, 0), (1, 1, 64, 4000, 64, 64, 0.1, 0, 2),
                  (1, 1, 64, 4000, 60, 64, 0.1, 0, 0), (1, 1, 64, 4000, 32, 32, 0.1, 0, 0), (1, 1, 64, 4000, 136, 136, 0.1, 0, 0)):
        assert need(0, *shape) == 0 and need(1, *shape) == 0
    n = ctypes.c_int64()
    assert lib.dlt_flash_workspace(L.FlashShape(1, 1, 8, 16, 64, 64, 1.0, 1, 0), 0, ctypes.byref(n)) == 1   # causal, Lq != Lk
    assert lib.dlt_flash_workspace(L.FlashShape(1, 1, 8, 16, 64, 64, 1.0, 0, 0), 0, None) == 1
    one, st4, st3 = ctypes.c_void_p(16), (ctypes.c_int64 * 4)(4096, 4096, 64, 1), (ctypes.c_int64 * 3)(64, 64, 1)
    for ws, size, word in ((16, 100, b"needed"), (20, 1 << 30, b"aligned")):
        rc = lib.dlt_flash_fwd_ws(one, st4, one, st4, one, st4, one, st4, one, st3, L.FlashShape(1, 1, 64, 4000, 64, 64, 0.1, 0, 0), ctypes.c_void_p(ws), size, None)
        assert rc == 1 and word in lib.dlt_last_error()
