"""CPU: the C-ABI library loads, exports exactly what include/mi355_kernels.h declares, and the
Python host surface keeps the reference's preconditions and error convention.  No kernel is
launched here."""
import ctypes
import os
import re

import pytest
import torch

import triton_amd
from triton_amd import _lib, ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = open(os.path.join(ROOT, "include", "mi355_kernels.h")).read()


def declared_functions():
    text = re.sub(r"/\*.*?\*/", "", HEADER, flags=re.S)
    return sorted(set(re.findall(r"\b(mi355_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = declared_functions()
    for n in ("mi355_gemm", "mi355_mx_gemm", "mi355_attn_fwd", "mi355_attn_bwd_preprocess", "mi355_attn_bwd",
              "mi355_dequant", "mi355_query", "mi355_strerror"):
        assert n in names


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    for n in declared_functions():
        assert hasattr(lib, n), f"{n} declared in the header but not exported"


def test_binding_table_matches_header():
    assert sorted(_lib.SIGNATURES) == declared_functions()


def test_header_is_plain_c():
    # the boundary carries no torch / C++ types: compile the header as C
    import subprocess, tempfile
    with tempfile.TemporaryDirectory() as d:
        src = os.path.join(d, "t.c")
        open(src, "w").write('#include "mi355_kernels.h"\nint main(void){return MI355_OK;}\n')
        subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"), "-c", src,
                        "-o", os.path.join(d, "t.o")], check=True)


def test_strerror_and_argument_rejection_without_gpu():
    lib = _lib.load()
    assert lib.mi355_strerror(0) == b"ok"
    assert b"invalid" in lib.mi355_strerror(-1)
    # null pointers are rejected before any device work
    assert lib.mi355_gemm(None, None, None, 4, 4, 4, 4, 1, 4, 1, 4, 1, 0, 0, None, None, 0, None) == -1
    assert lib.mi355_query(12345) == -1


def test_products_with_rows_too_far_apart_for_the_tile_kernels_copy_them():
    # rows of B 64 MiB apart (row major) or 8 MiB (K major) are beyond the kernels' lane offsets: a B that would otherwise
    # stay in place beside the copy of an unaligned A is copied too, as only those kernels know that its rows end before A's padding
    lib = _lib.load()

    def need(sbk, sbn, K=73, b=1 << 21):
        return lib.mi355_gemm_workspace(1 << 20, b, 2048, 2048, K, K, 1, sbk, sbn, _lib.BF16)
    a_copy = 256 * 2048
    assert need(2048, 1) == need((1 << 25) - 8, 1) == a_copy
    assert need(1 << 25, 1) == a_copy + 4096 * 128            # (B's copy has the rows of zeros beyond K)
    assert need(1 << 40, 1) == a_copy + 4096 * 128
    assert need(1, 1 << 22) == need(1, 80) == 2 * a_copy      # (a K-major B is always copied here: its rows are not whole chunks)


def _workspace(M, N, K, dtype, kmajor=True, ldb=None):
    """Bytes that matmul asks for (256 CUs, aligned operands): copies of unaligned rows and slices of a split K."""
    b = (1, ldb or K) if kmajor else (ldb or N, 1)
    return _lib.load().mi355_gemm_workspace(1 << 20, 1 << 21, M, N, K, K, 1, *b, dtype)


def test_fp32_products_are_split_where_that_shortens_the_fullest_cu():
    # tiles of 128x128 per CU times K steps per slice: no split of few steps or of nearly a round of tiles, remainders taken account of
    for M, N, K, slices in ((2048, 1920, 256, 0), (2048, 1920, 2048, 0), (1536, 1536, 512, 0), (1536, 1536, 1024, 3), (1024, 1024, 1024, 4),
                            (1024, 1408, 4096, 8), (512, 512, 8192, 16)):
        assert _workspace(M, N, K, _lib.F32) == slices * 4 * M * N, (M, N, K)


def test_rows_are_not_copied_for_a_single_short_step():
    # K below 48 with rows of C that are no whole groups of four: the kernel of any strides (B's rows are not 16-byte chunks)
    assert _workspace(4024, 5214, 16, _lib.F8E4M3, False, 5230) == 0
    assert _workspace(5246, 2775, 30, _lib.F16, False) == 0
    assert _workspace(5248, 1792, 28, _lib.F8E4M3, False) > 0
    assert _workspace(2084, 2092, 63, _lib.F8E4M3, False) > 0


def test_few_rows_are_split_where_that_pays_for_the_second_launch():
    for M, N, K, slices in ((16, 320, 4704, 0), (64, 2048, 2048, 0), (16, 8192, 8192, 0), (64, 8192, 8192, 2), (32, 4096, 4096, 4)):
        assert _workspace(M, N, K, _lib.F16) == slices * 4 * M * N, (M, N, K)


def test_matmul_preconditions_match_reference_messages():
    a = torch.zeros(4, 8, dtype=torch.float16)
    b = torch.zeros(6, 4, dtype=torch.float16)
    with pytest.raises(AssertionError, match="Incompatible dimensions"):   # 03:332
        triton_amd.matmul(a, b)
    with pytest.raises(AssertionError, match="Matrix A must be contiguous"):  # 03:333
        triton_amd.matmul(torch.zeros(8, 4, dtype=torch.float16).t(), torch.zeros(8, 4, dtype=torch.float16))
    with pytest.raises(AssertionError, match="Incompatible dtypes"):       # semantic.py:1355 / 09:121
        triton_amd.matmul(a, torch.zeros(8, 4, dtype=torch.bfloat16))


def test_cpu_tensor_is_a_value_error_like_the_reference_launcher():
    # third_party/amd/backend/driver.py:313-317
    a = torch.zeros(4, 8, dtype=torch.float16)
    b = torch.zeros(8, 4, dtype=torch.float16)
    with pytest.raises(ValueError, match="cannot be accessed from Triton"):
        triton_amd.matmul(a, b)


def test_attention_preconditions():
    q = torch.zeros(1, 1, 128, 48, dtype=torch.float16)
    with pytest.raises(AssertionError):      # HEAD_DIM in {16,32,64,128,256} (06:447)
        triton_amd.attention(q, q, q, True, 0.5)
    k = torch.zeros(1, 1, 128, 64, dtype=torch.float16)
    with pytest.raises(AssertionError):      # equal head dims (06:446)
        triton_amd.attention(torch.zeros(1, 1, 128, 32, dtype=torch.float16), k, k, True, 0.5)


def test_status_to_exception_mapping():
    _lib.check(0, "x")
    with pytest.raises(RuntimeError, match=r"Triton Error \[HIP\]"):   # driver.py:258-269
        _lib.check(1, "x")
    with pytest.raises(ValueError):
        _lib.check(-3, "x")


def test_dtype_names_of_reinterpreted_tensors():
    class Wrapped:   # stands in for triton.reinterpret(t, tl.float8e4nv) (jit.py:895-938)
        class dtype:
            name = "fp8e4nv"
    assert ops._abi_dtype(Wrapped()) == _lib.F8E4M3
    assert ops._abi_dtype(torch.zeros(1, dtype=torch.bfloat16)) == _lib.BF16


def test_launch_record_matches_the_tutorial_formulas():
    # python/tutorials/09-persistent-matmul.py:34-45 and 06-fused-attention.py:630-634, evaluated lazily
    from triton_amd import hooks

    calls = []

    def counted(*args):
        calls.append(args)
        return hooks.matmul_launch_metadata(*args)

    md = hooks.LaunchMetadata({"name": "k", "stream": 7})
    md.add(counted, ("k", 16, 8192, 8192, 1))
    assert calls == []                       # nothing evaluated until a hook asks
    rec = md.get()
    assert rec == {"name": "k [M=16, N=8192, K=8192]", "stream": 7, "flops8": 2.0 * 16 * 8192 * 8192,
                   "bytes": 16 * 8192 + 8192 * 8192}
    md.get()
    assert len(calls) == 1                   # and only once
    rec = hooks.attention_launch_metadata("a", 4, 32, 4096, 128, False, 2)
    assert rec["flops16"] == 2 * 2.0 * 4 * 32 * 4096 * 4096 * 128
    assert hooks.enter("x", 0, hooks.matmul_launch_metadata, ("x", 1, 1, 1, 2)) is None   # no hook set
