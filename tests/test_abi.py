"""The C ABI without a GPU: the library loads, exports every symbol the header
declares, and every validation error path returns its code before any HIP call."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gguf_hip.h")


def _header():
    with open(HEADER, encoding="utf-8") as f:
        return f.read()


def _declared_functions():
    return re.findall(r"^\s*(?:int|int64_t|const char \*)\s*\*?\s*(gguf_hip_\w+)\s*\(", _header(),
                      re.M)


def _defines():
    return {m.group(1): int(m.group(2).strip("()"))
            for m in re.finditer(r"#define\s+(GGUF_HIP_\w+)\s+(\(?-?\d+\)?)", _header())}


@pytest.fixture(scope="module")
def lib(pkg):
    from importlib import import_module
    native = import_module("artifex-assistantv5_amd._native")
    if not os.path.exists(native.LIB_PATH):
        import_module("artifex-assistantv5_amd.build").build()
    return native.load_library()


@pytest.fixture(scope="module")
def native(pkg):
    from importlib import import_module
    return import_module("artifex-assistantv5_amd._native")


def test_exports_every_declared_symbol(lib, native):
    names = _declared_functions()
    assert len(names) == 24, names
    for n in names:
        assert hasattr(lib, n), n
        assert n in native.SIGNATURES, n
    assert set(native.SIGNATURES) == set(names)


def test_constants_match_header(native):
    d = _defines()
    assert d["GGUF_HIP_ABI_VERSION"] == native.ABI_VERSION
    assert d["GGUF_HIP_ERR_TYPE"] == native.ERR_TYPE
    assert d["GGUF_HIP_ERR_SHAPE"] == native.ERR_SHAPE
    assert d["GGUF_HIP_ERR_NULL"] == native.ERR_NULL
    assert d["GGUF_HIP_ERR_ALIGN"] == native.ERR_ALIGN
    assert d["GGUF_HIP_ERR_DTYPE"] == native.ERR_DTYPE
    assert d["GGUF_HIP_ERR_BYTES"] == native.ERR_BYTES
    assert d["GGUF_HIP_ERR_HIP"] == native.ERR_HIP
    assert d["GGUF_HIP_VARIANT_DECODE"] == native.VARIANT_DECODE
    assert d["GGUF_HIP_VARIANT_GEMM"] == native.VARIANT_GEMM
    assert d["GGUF_HIP_DECODE_MAX_M"] == native.DECODE_MAX_M
    assert d["GGUF_HIP_NOALLOC_ATTENTION_BYTES"] == native.NOALLOC_ATTENTION_BYTES
    assert (d["GGUF_HIP_Q8_0"], d["GGUF_HIP_Q4_K"], d["GGUF_HIP_Q5_K"],
            d["GGUF_HIP_Q6_K"]) == (8, 12, 13, 14)
    assert (d["GGUF_HIP_Q4_0"], d["GGUF_HIP_Q5_0"], d["GGUF_HIP_IQ4_NL"],
            d["GGUF_HIP_IQ4_XS"]) == (2, 6, 20, 23)
    assert (d["GGUF_HIP_IQ2_XXS"], d["GGUF_HIP_IQ2_XS"], d["GGUF_HIP_IQ3_XXS"], d["GGUF_HIP_IQ3_S"],
            d["GGUF_HIP_IQ2_S"], d["GGUF_HIP_IQ1_M"]) == (16, 17, 18, 21, 22, 29)


def test_one_row_needs_no_workspace_up_to_the_limit(lib, native, pkg):
    """The host asks for no workspace for one row of up to ONE_SHOT_MAX_K elements."""
    limit = native.ONE_SHOT_MAX_K
    assert _defines()["GGUF_HIP_ONE_SHOT_MAX_K"] == limit
    for t in (2, 6, 8, 10, 11, 12, 13, 14, 16, 17, 18, 20, 21, 22, 23, 29):
        for x_type in (0, 1):
            for n in (1, 4096, 151936):
                for k in (256, 4096, limit - 256, limit):
                    assert lib.gguf_hip_matmul_workspace(t, x_type, n, k, 1) == 0, (t, n, k)
    for t in (16, 17, 18, 21, 22, 29):
        assert lib.gguf_hip_matmul_workspace(t, 0, 4096, limit + 256, 1) > 0


def test_grid_types_contract(lib, native):
    """IQ2_XXS .. IQ1_M: no workspace needed for the decode variant up to
    K = 16384 (M = 1 asks for none, M >= 2 for an optional one); beyond it a
    workspace is required, and the fused kernels stop there as for the other
    types.  Fake (aligned, never dereferenced) pointers: every check below
    fails before any HIP call."""
    x, w, y = 0x10000, 0x20000, 0x30000
    for t in (16, 17, 18, 21, 22, 29):
        for xt in (0, 1):
            assert lib.gguf_hip_matmul_workspace(t, xt, 64, 512, 1) == 0
            assert lib.gguf_hip_matmul_workspace(t, xt, 64, 16384, 1) == 0
            for m in (5, 40):
                assert lib.gguf_hip_matmul_workspace(t, xt, 64, 512, m) > 0
            assert lib.gguf_hip_matmul_workspace(t, xt, 64, 16640, 1) > 0
        assert lib.gguf_hip_matmul(x, 0, 16640, w, t, 64, 16640, y, 64, 1, None) == native.ERR_SHAPE
        assert "needs a workspace" in native.last_error(lib)
        need = lib.gguf_hip_matmul_workspace(t, 0, 64, 16640, 3)
        assert lib.gguf_hip_matmul_ws(x, 0, 16640, w, t, 64, 16640, y, 64, 3, 0, 0x40000,
                                      need - 16, None) == native.ERR_SHAPE
        # fused kernels exist for these types too, up to K = 16384 like the others
        assert lib.gguf_hip_matmul_fused(x, w, t, 64, 16640, y, 0, None, ctypes.c_float(0.0), 0,
                                         None) == native.ERR_SHAPE
        assert "above 16384" in native.last_error(lib)
    assert (lib.gguf_hip_matmul_workspace(12, 0, 64, 512, 1), lib.gguf_hip_matmul_workspace(
        20, 0, 64, 512, 1)) == (0, 0)


def test_abi_version(lib):
    assert lib.gguf_hip_abi_version() == 18


def test_type_traits(lib, native):
    b, s = ctypes.c_int(), ctypes.c_int()
    assert lib.gguf_hip_type_traits(12, ctypes.byref(b), ctypes.byref(s)) == 0
    assert (b.value, s.value) == (256, 144)
    assert lib.gguf_hip_type_traits(99, ctypes.byref(b), ctypes.byref(s)) == native.ERR_TYPE
    assert "Unsupported ggml type 99" in native.last_error(lib)


def test_byte_queries_agree_with_python(lib, pkg):
    for t in (2, 6, 8, 10, 11, 12, 13, 14, 20, 23, 16, 17, 18, 21, 22, 29):
        for k in (256, 512, 1024, 4096, 14336):
            assert lib.gguf_hip_tile_bytes(t, 7, k) == 16 * pkg.tile_row_bytes(t, k)
            assert lib.gguf_hip_tile_bytes(t, 33, k) == pkg.tiled_bytes(t, 33, k)
            assert lib.gguf_hip_raw_bytes(t, 7, k) == pkg.ggml_tensor_bytes(t, [k, 7])
    assert lib.gguf_hip_tile_bytes(3, 1, 256) == -1    # Q4_1: known type, no kernel
    assert lib.gguf_hip_tile_bytes(8, 1, 48) == -2


def test_repack_errors(lib, native):
    raw_bytes = 2 * 144
    tiled = 16 * raw_bytes                 # one row occupies a whole 16-row tile
    # byte length mismatch (assertBytes, gguf-dequant.ts:678-680)
    assert lib.gguf_hip_repack(None, raw_bytes - 1, 12, 1, 512, None, tiled, None) == native.ERR_BYTES
    assert "byteLength 287 != expected 288" in native.last_error(lib)
    assert lib.gguf_hip_repack(None, raw_bytes, 12, 1, 512, None, 288, None) == native.ERR_BYTES
    assert lib.gguf_hip_repack(None, raw_bytes, 12, 1, 512, None, tiled, None) == native.ERR_NULL
    assert lib.gguf_hip_repack(0x1000, raw_bytes, 12, 1, 512, 0x1008, tiled, None) == native.ERR_ALIGN
    assert lib.gguf_hip_repack(0x1000, 10, 99, 1, 512, 0x1000, tiled, None) == native.ERR_TYPE
    assert lib.gguf_hip_repack(0x1000, 10, 12, 1, 300, 0x1000, tiled, None) == native.ERR_SHAPE
    assert lib.gguf_hip_repack(None, 0, 12, 0, 512, None, 0, None) == 0     # empty: no-op


def test_dequant_errors(lib, native):
    assert lib.gguf_hip_dequant(None, 12, 1, 512, None, 512, None) == native.ERR_NULL
    assert lib.gguf_hip_dequant(0x1004, 12, 1, 512, 0x2000, 512, None) == native.ERR_ALIGN
    assert lib.gguf_hip_dequant(0x1000, 12, 1, 512, 0x2002, 512, None) == native.ERR_ALIGN
    assert lib.gguf_hip_dequant(0x1000, 12, 2, 512, 0x2000, 256, None) == native.ERR_SHAPE
    assert lib.gguf_hip_dequant(0x1000, 3, 1, 512, 0x2000, 512, None) == native.ERR_TYPE
    assert "no kernel for ggml type 3" in native.last_error(lib)
    assert lib.gguf_hip_dequant(0x1000, 14, 1, 100, 0x2000, 512, None) == native.ERR_SHAPE
    assert "not divisible by block size 256" in native.last_error(lib)
    assert lib.gguf_hip_dequant_raw(None, 8, 33, None, None) == native.ERR_SHAPE
    assert lib.gguf_hip_dequant_raw(None, 8, 64, None, None) == native.ERR_NULL
    assert lib.gguf_hip_dequant_raw(None, 8, 0, None, None) == 0


def test_get_rows_errors(lib, native):
    gr = lib.gguf_hip_get_rows
    raw, ids, out = 0x1000, 0x2000, 0x3000
    assert gr(raw, 3, 4, 512, ids, 1, out, 512, None) == native.ERR_TYPE
    assert gr(raw, 12, 4, 300, ids, 1, out, 512, None) == native.ERR_SHAPE
    assert gr(raw, 12, -1, 512, ids, 1, out, 512, None) == native.ERR_SHAPE
    assert gr(raw, 12, 4, 512, ids, 2, out, 256, None) == native.ERR_SHAPE     # ldo < K
    assert gr(None, 12, 4, 512, ids, 1, out, 512, None) == native.ERR_NULL
    assert gr(raw, 12, 4, 512, ids + 4, 1, out, 512, None) == native.ERR_ALIGN
    assert gr(raw, 12, 4, 512, ids, 1, out + 2, 512, None) == native.ERR_ALIGN
    assert gr(None, 12, 4, 512, None, 0, None, 512, None) == 0                 # no ids: no-op


def test_matmul_errors(lib, native):
    mm = lib.gguf_hip_matmul_variant
    x, w, y = 0x10000, 0x20000, 0x30000
    assert mm(x, 2, 512, w, 12, 8, 512, y, 8, 1, 0, None) == native.ERR_DTYPE
    assert mm(x, 0, 512, w, 12, 8, 512, y, 8, 1, 9, None) == native.ERR_SHAPE    # bad variant
    assert "unknown kernel variant 9" in native.last_error(lib)
    assert mm(x, 0, 512, w, 12, 8, 512, y, 8, 1, -1, None) == native.ERR_SHAPE
    assert mm(x, 0, 512, w, 3, 8, 512, y, 8, 1, 0, None) == native.ERR_TYPE      # Q4_1
    assert mm(x, 0, 512, w, 12, 8, 500, y, 8, 1, 0, None) == native.ERR_SHAPE
    assert mm(None, 0, 512, w, 12, 8, 512, y, 8, 1, 0, None) == native.ERR_NULL
    assert mm(x + 4, 0, 512, w, 12, 8, 512, y, 8, 1, 0, None) == native.ERR_ALIGN
    assert mm(x, 0, 513, w, 12, 8, 512, y, 8, 2, 0, None) == native.ERR_ALIGN    # row stride
    assert mm(x, 0, 512, w + 8, 12, 8, 512, y, 8, 1, 0, None) == native.ERR_ALIGN
    assert mm(x, 0, 512, w, 12, 8, 512, y + 2, 8, 1, 0, None) == native.ERR_ALIGN
    assert mm(x, 0, 256, w, 12, 8, 512, y, 8, 2, 0, None) == native.ERR_SHAPE    # ldx < K
    assert mm(x, 0, 512, w, 12, 8, 512, y, 4, 2, 0, None) == native.ERR_SHAPE    # ldy < N
    assert mm(x, 0, 512, w, 12, -1, 512, y, 8, 1, 0, None) == native.ERR_SHAPE
    # empty problems are no-ops and touch nothing
    assert mm(None, 0, 512, None, 12, 8, 512, None, 8, 0, 0, None) == 0
    assert lib.gguf_hip_matmul(None, 0, 512, None, 12, 0, 512, None, 8, 4, None) == 0


def test_python_error_mapping(lib, native):
    with pytest.raises(NotImplementedError):
        native.check(native.ERR_TYPE, lib)
    for code in (native.ERR_SHAPE, native.ERR_NULL, native.ERR_ALIGN, native.ERR_DTYPE,
                 native.ERR_BYTES):
        with pytest.raises(ValueError):
            native.check(code, lib)
    with pytest.raises(native.GGUFHipError):
        native.check(native.ERR_HIP, lib)
    assert native.check(0, lib) == 0


def test_last_error_is_thread_local(lib, native):
    import threading
    assert lib.gguf_hip_tile_bytes(99, 1, 256) == native.ERR_TYPE
    seen = {}

    def other():
        seen["msg"] = lib.gguf_hip_last_error()

    th = threading.Thread(target=other)
    th.start()
    th.join()
    assert seen["msg"] in (b"", None)
    assert "Unsupported" in native.last_error(lib)


def test_single_hip_runtime_mapped(lib, native):
    assert len(native._hip_runtimes_mapped()) <= 1


def test_glue_errors(lib, native):
    a, b, c = 0x10000, 0x20000, 0x30000
    assert lib.gguf_hip_rmsnorm(a, b, 1e-6, c, 1, 4094, None) == native.ERR_SHAPE   # n % 4
    assert lib.gguf_hip_rmsnorm(a, b, -1.0, c, 1, 4096, None) == native.ERR_SHAPE
    assert lib.gguf_hip_rmsnorm(None, b, 1e-6, c, 1, 4096, None) == native.ERR_NULL
    assert lib.gguf_hip_rmsnorm(a + 4, b, 1e-6, c, 1, 4096, None) == native.ERR_ALIGN
    assert lib.gguf_hip_rmsnorm(None, None, 1e-6, None, 0, 4096, None) == 0         # no rows
    assert lib.gguf_hip_add_rmsnorm(a, b, b, 1e-6, a, 1, 4096, None) == native.ERR_SHAPE
    assert "aliases" in native.last_error(lib)
    assert lib.gguf_hip_swiglu(a, b, 1, 14338, None) == native.ERR_SHAPE
    assert lib.gguf_hip_swiglu(a, b + 8, 1, 14336, None) == native.ERR_ALIGN
    att = lib.gguf_hip_attention_decode
    wk = 0x40000
    assert att(a, b, c, c, a, a, b, 32, 5, 128, 512, wk, None) == native.ERR_SHAPE  # 32 % 5
    assert att(a, b, c, c, a, a, b, 32, 2, 128, 512, wk, None) == native.ERR_SHAPE  # grp 16 > 8
    assert att(a, b, c, c, a, a, b, 32, 8, 96, 512, wk, None) == native.ERR_SHAPE   # head_dim
    assert "head_dim 96" in native.last_error(lib)
    assert att(a, b, c, c, a, a, b, 32, 8, 128, 0, wk, None) == native.ERR_SHAPE
    assert att(None, b, c, c, a, a, b, 32, 8, 128, 512, wk, None) == native.ERR_NULL
    assert att(a, b, c, c, a, a, b, 32, 8, 128, 512, None, None) == native.ERR_NULL
    assert att(a + 4, b, c, c, a, a, b, 32, 8, 128, 512, wk, None) == native.ERR_ALIGN
    # workspace: 8 KV heads x 8 slot ranges of 64 x 4 query heads x (128 + 4) floats
    # records [nkv][S][grp][hd + 4] floats, then nkv counters (16-byte rounded)
    assert lib.gguf_hip_attention_workspace(32, 8, 128, 512) == 8 * 8 * 4 * 132 * 4 + 32
    assert lib.gguf_hip_attention_workspace(4, 2, 64, 65) == 2 * 2 * 2 * 68 * 4 + 16
    assert lib.gguf_hip_attention_workspace(32, 8, 100, 512) == native.ERR_SHAPE
    # the entry point without a workspace: same checks, plus the size of its own array
    na = lib.gguf_hip_attention_decode_noalloc
    assert na(a, b, c, c, a, a, b, 32, 5, 128, 512, None) == native.ERR_SHAPE
    assert na(a, b, c, c, a, a, None, 32, 8, 128, 512, None) == native.ERR_NULL    # out required
    assert na(a + 4, b, c, c, a, a, b, 32, 8, 128, 512, None) == native.ERR_ALIGN
    big = lib.gguf_hip_attention_workspace(64, 8, 128, 65536)
    assert big > native.NOALLOC_ATTENTION_BYTES
    assert na(a, b, c, c, a, a, b, 64, 8, 128, 65536, None) == native.ERR_SHAPE
    assert "noalloc" in native.last_error(lib)
    # prefill attention: qkv row 32*128 + 2*8*128 = 6144 floats, out row 4096
    pf = lib.gguf_hip_attention_prefill
    assert pf(a, 6144, b, 128, c, c, a, a, b, 4096, 32, 5, 128, 512, None) == native.ERR_SHAPE
    assert pf(a, 6144, b, 128, c, c, a, a, b, 4096, 32, 8, 96, 512, None) == native.ERR_SHAPE
    assert pf(a, 6140, b, 128, c, c, a, a, b, 4096, 32, 8, 128, 512, None) == native.ERR_SHAPE
    assert pf(a, 6146, b, 128, c, c, a, a, b, 4096, 32, 8, 128, 512, None) == native.ERR_SHAPE
    assert pf(a, 6144, b, 128, c, c, a, a, b, 4092, 32, 8, 128, 512, None) == native.ERR_SHAPE
    assert "ldqkv" in native.last_error(lib)
    assert pf(a, 6144, b, -1, c, c, a, a, b, 4096, 32, 8, 128, 512, None) == native.ERR_SHAPE
    assert pf(None, 6144, None, 0, None, None, None, None, None, 4096, 32, 8, 128, 512,
              None) == 0                                                      # no rows
    assert pf(a, 6144, b, 4, c, c, a, a, None, 4096, 32, 8, 128, 512, None) == native.ERR_NULL
    assert pf(a, 6144, b + 4, 4, c, c, a, a, b, 4096, 32, 8, 128, 512, None) == native.ERR_ALIGN
    assert pf(a, 6144, b, 4, c + 4, c, a, a, b, 4096, 32, 8, 128, 512, None) == native.ERR_ALIGN
    assert pf(a, 6144, b, 4, c, c, a, a, b + 4, 4096, 32, 8, 128, 512, None) == native.ERR_ALIGN
    assert lib.gguf_hip_argmax_workspace() > 0
    assert lib.gguf_hip_argmax(a, 0, b, c, None) == native.ERR_SHAPE
    assert lib.gguf_hip_argmax(a, 10, b + 4, c, None) == native.ERR_ALIGN
    assert lib.gguf_hip_argmax(a, 10, b, None, None) == native.ERR_NULL


def test_attn_merge_errors(lib, native):
    f = lib.gguf_hip_matmul_attn_merge
    wk, pos, w, y = 0x10000, 0x20000, 0x30000, 0x40000
    assert f(wk, pos, 32, 5, 128, 512, w, 12, 64, y, 1, None) == native.ERR_SHAPE   # 32 % 5
    assert f(wk, pos, 32, 8, 96, 512, w, 12, 64, y, 1, None) == native.ERR_SHAPE    # head_dim
    assert f(wk, pos, 32, 8, 128, 0, w, 12, 64, y, 1, None) == native.ERR_SHAPE     # max_seq
    assert f(wk, pos, 32, 8, 128, 512, w, 3, 64, y, 1, None) == native.ERR_TYPE
    assert f(wk, pos, 3, 1, 64, 512, w, 12, 64, y, 1, None) == native.ERR_SHAPE     # K=192 % 256
    assert f(wk, pos, 32, 8, 128, 512, w, 12, 64, y, 2, None) == native.ERR_SHAPE   # SwiGLU epi
    assert "epilogue 2" in native.last_error(lib)
    for max_seq in (512, 4096):
        assert f(wk, pos, 64, 8, 256, max_seq, w, 12, 64, y, 1, None) == native.ERR_SHAPE   # K=16384
    assert "no merge kernel" in native.last_error(lib)
    assert f(None, pos, 32, 8, 128, 512, w, 12, 64, y, 1, None) == native.ERR_NULL
    assert f(wk, None, 32, 8, 128, 512, w, 12, 64, y, 1, None) == native.ERR_NULL
    assert f(wk + 4, pos, 32, 8, 128, 512, w, 12, 64, y, 1, None) == native.ERR_ALIGN
    assert f(wk, pos + 4, 32, 8, 128, 512, w, 12, 64, y, 1, None) == native.ERR_ALIGN
    assert f(None, None, 32, 8, 128, 512, None, 12, 0, None, 0, None) == 0          # N = 0


def test_fused_matmul_errors(lib, native):
    f = lib.gguf_hip_matmul_fused
    x, w, y, nw = 0x10000, 0x20000, 0x30000, 0x40000
    assert f(x, w, 12, 64, 4096, y, 3, nw, 1e-6, 0, None) == native.ERR_SHAPE      # prologue
    assert f(x, w, 12, 64, 32768, y, 0, None, 0.0, 0, None) == native.ERR_SHAPE    # K > 16384
    assert "16384" in native.last_error(lib)
    assert f(x, w, 12, 64, 4096, y, 1, None, 1e-6, 0, None) == native.ERR_NULL     # no norm weight
    assert f(x, w, 12, 64, 4096, y, 1, nw, -1.0, 0, None) == native.ERR_SHAPE
    assert f(x + 4, w, 12, 64, 4096, y, 0, None, 0.0, 0, None) == native.ERR_ALIGN
    assert f(x, w, 3, 64, 4096, y, 0, None, 0.0, 0, None) == native.ERR_TYPE
    assert f(x, w, 12, 64, 4096, y, 0, None, 0.0, 3, None) == native.ERR_SHAPE      # epilogue
    assert f(x, w, 12, 48, 4096, y, 0, None, 0.0, 2, None) == native.ERR_SHAPE      # SwiGLU: N % 32
    assert f(x, w, 12, 0, 4096, y, 2, None, 0.0, 1, None) == 0                     # N = 0: no-op
    d = _defines()
    assert (d["GGUF_HIP_PROLOGUE_NONE"], d["GGUF_HIP_PROLOGUE_RMSNORM"],
            d["GGUF_HIP_PROLOGUE_SWIGLU"]) == (native.PROLOGUE_NONE, native.PROLOGUE_RMSNORM,
                                               native.PROLOGUE_SWIGLU)
    assert (d["GGUF_HIP_EPILOGUE_STORE"], d["GGUF_HIP_EPILOGUE_ACCUMULATE"],
            d["GGUF_HIP_EPILOGUE_SWIGLU"]) == (native.EPILOGUE_STORE, native.EPILOGUE_ACCUMULATE,
                                               native.EPILOGUE_SWIGLU)
