"""CPU-side checks of the drop-in boundary: the C ABI exports what the header declares,
argument validation works without a GPU, and the Python modules keep the reference's
constructor/attribute/error contract.  No kernel is launched here."""

import ctypes
import re
from pathlib import Path

import numpy as np
import pytest
import torch

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "q4_linear.h"


def declared_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(q4_[a-z_0-9]+)\s*\(", text)))


def test_header_functions_are_exported_and_bound(pkg):
    lib = pkg._lib.load()
    names = declared_functions()
    assert {"q4_dequant", "q4_linear", "q4_linear_ex", "q4_gemv_tuned", "q4_linear_gate_up", "q4_act_mul", "q4_workspace_bytes",
            "q4_select_path", "q4_last_error", "q4_abi_version"} <= set(names)
    for name in names:
        assert hasattr(lib, name), f"{name} declared in q4_linear.h but not exported"
        assert name in pkg._lib.SIGNATURES, f"{name} has no ctypes signature"
    assert sorted(pkg._lib.SIGNATURES) == names
    assert lib.q4_abi_version() == 1


def test_header_constants_match_binding(pkg):
    text = HEADER.read_text()
    consts = dict(re.findall(r"#define\s+(Q4_[A-Z_0-9]+)\s+\(?(-?\d+)\)?", text))
    L = pkg._lib
    assert int(consts["Q4_LAYOUT_GPTQ"]) == L.LAYOUT_GPTQ and int(consts["Q4_LAYOUT_AWQ"]) == L.LAYOUT_AWQ
    assert int(consts["Q4_DTYPE_F16"]) == L.DTYPE_F16 and int(consts["Q4_DTYPE_BF16"]) == L.DTYPE_BF16
    assert int(consts["Q4_PATH_GEMV"]) == L.PATH_GEMV and int(consts["Q4_PATH_GEMM"]) == L.PATH_GEMM
    assert int(consts["Q4_PATH_GENERIC"]) == L.PATH_GENERIC
    assert int(consts["Q4_WORKSPACE_COUNTER_BYTES"]) == L.WORKSPACE_COUNTER_BYTES
    assert int(consts["Q4_ERR_INVALID_ARGUMENT"]) == L.ERR_INVALID_ARGUMENT
    assert int(consts["Q4_ERR_UNSUPPORTED"]) == L.ERR_UNSUPPORTED
    assert int(consts["Q4_ERR_WORKSPACE"]) == L.ERR_WORKSPACE


def _weight(pkg, K, N, gs, layout=0, g_idx=False):
    """A q4_weight with fake non-null pointers: only used on paths that never dereference."""
    G = max(1, K // gs) if gs > 0 else 1
    return pkg._lib.Q4Weight(0x1000, 0x2000, 0x3000, 0x4000 if g_idx else None, K, N, gs, G, layout)


def test_argument_validation_without_gpu(pkg):
    lib = pkg._lib.load()
    L = pkg._lib
    assert lib.q4_dequant(None, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert b"null q4_weight" in lib.q4_last_error()
    w = _weight(pkg, 4096, 4100, 128)  # N not a multiple of 8
    assert lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, 1, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert b"multiples of 8" in lib.q4_last_error()
    w = _weight(pkg, 4096, 4096, 128, layout=7)
    assert lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, 1, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    w = _weight(pkg, 4096, 4096, 128)
    assert lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, 1, 9, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert b"dtype" in lib.q4_last_error()
    assert lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, -1, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    # groups must cover K when there is no g_idx
    w = pkg._lib.Q4Weight(0x1000, 0x2000, 0x3000, None, 4096, 4096, 128, 8, 0)
    assert lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, 1, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert b"do not cover" in lib.q4_last_error()
    # AWQ has no act-order
    w = _weight(pkg, 4096, 4096, 128, layout=1, g_idx=True)
    assert lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, 1, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    # decode path without the workspace it needs is refused before any launch
    w = _weight(pkg, 4096, 4096, 128)
    assert lib.q4_linear_ex(ctypes.byref(w), 0x10, None, 0x20, 1, 0, None, 0, L.PATH_GEMV, None) == L.ERR_WORKSPACE
    assert b"workspace" in lib.q4_last_error()
    # empty problems succeed without touching anything
    w = _weight(pkg, 4096, 0, 128)
    assert lib.q4_linear(ctypes.byref(w), None, None, None, 4, 0, None, 0, None) == 0
    w = _weight(pkg, 4096, 4096, 128)
    assert lib.q4_linear(ctypes.byref(w), None, None, None, 0, 0, None, 0, None) == 0


def test_moe_argument_validation_without_gpu(pkg):
    """The grouped entry points reject bad arguments before anything is launched."""
    import ctypes

    lib = pkg._lib.load()
    L = pkg._lib

    def moe(K, N, gs, experts=8, layout=0, g_idx=False, strides=None):
        e0 = _weight(pkg, K, N, gs, layout, g_idx)
        G = max(1, K // gs)
        st = strides or ((K // 8) * N, G * (N // 8), G * N, K)
        return L.Q4MoeWeight(e0, experts, *st)

    assert int(L.DTYPE_F32) == 2
    # routing: experts and topk limits, null outputs
    assert lib.q4_moe_route(0x10, 2, 4, 300, 2, 1, 0x20, 0x30, 0x40, 0x50, 0x60, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_route(0x10, 2, 4, 8, 9, 1, 0x20, 0x30, 0x40, 0x50, 0x60, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_route(0x10, 2, 4, 8, 2, 1, None, 0x30, 0x40, 0x50, 0x60, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_route(0x10, 7, 4, 8, 2, 1, 0x20, 0x30, 0x40, 0x50, 0x60, None) == L.ERR_INVALID_ARGUMENT
    assert b"gating dtype" in lib.q4_last_error()
    # grouped linear: null weight, bad geometry, strides smaller than an expert, AWQ with g_idx
    assert lib.q4_moe_linear(None, 0x10, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    w = moe(4096, 4100, 128)
    assert lib.q4_moe_linear(ctypes.byref(w), 0x10, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    w = moe(4096, 4096, 128, strides=(100, 100, 100, 100))
    assert lib.q4_moe_linear(ctypes.byref(w), 0x10, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert b"strides" in lib.q4_last_error()
    w = moe(4096, 4096, 128, layout=1, g_idx=True)
    assert lib.q4_moe_linear(ctypes.byref(w), 0x10, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    w = moe(4096, 4096, 128, experts=0)
    assert lib.q4_moe_linear(ctypes.byref(w), 0x10, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    w = moe(4096, 4096, 128)
    assert lib.q4_moe_linear(ctypes.byref(w), 0x10, None, 0x20, 0x30, 4, 2, 5, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_linear(ctypes.byref(w), None, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_linear(ctypes.byref(w), None, None, None, None, 0, 2, 0, None, 0, None) == 0  # no tokens
    # a shape no grouped kernel takes (K not a multiple of 64)
    w = moe(4104, 4096, 8)
    assert lib.q4_moe_linear(ctypes.byref(w), 0x10, None, 0x20, 0x30, 4, 2, 0, None, 0, None) == L.ERR_UNSUPPORTED
    # weighted sum
    assert lib.q4_moe_combine(0x10, 0x20, 0x30, 0x40, 4, 2, 4100, 0, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_combine(0x10, 0x20, 0x30, None, 4, 2, 4096, 0, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_moe_combine(None, None, None, None, 0, 2, 4096, 0, None) == 0
    # workspace: at least the counters; more when the decode plan splits K over workgroups
    w = moe(4096, 4096, 128)
    assert lib.q4_moe_workspace_bytes(ctypes.byref(w), 1, 2) >= L.WORKSPACE_COUNTER_BYTES
    assert lib.q4_moe_workspace_bytes(ctypes.byref(w), 1024, 2) >= L.WORKSPACE_COUNTER_BYTES
    assert lib.q4_moe_workspace_bytes(None, 1, 2) == 0


def test_workspace_sizing_covers_every_launch(pkg):
    """A workspace of the advertised size is never reported as too small, whatever kernel the
    dispatch takes (the launch itself fails here for want of a GPU, after the size check)."""
    import ctypes

    lib = pkg._lib.load()
    L = pkg._lib
    for layout, g_idx in ((0, False), (0, True), (1, False)):
        for K, N in [(14336, 4096), (4096, 28672), (4096, 4096), (11008, 4096), (8192, 1024), (5504, 512)]:
            for M in (1, 2, 3, 4, 8, 12, 16, 17, 32, 40, 64, 65, 200, 1000, 2048):
                for dt in (0, 1):
                    w = _weight(pkg, K, N, 128, layout, g_idx)
                    ws = lib.q4_workspace_bytes(M, K, N)
                    rc = lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, M, dt, 0x40, ws, None)
                    assert rc != L.ERR_WORKSPACE, (layout, g_idx, K, N, M, dt, lib.q4_last_error())
                    G = K // 128
                    mw = L.Q4MoeWeight(w, 8, (K // 8) * N, G * (N // 8), G * N, K)
                    ws = lib.q4_moe_workspace_bytes(ctypes.byref(mw), M, 2)
                    rc = lib.q4_moe_linear(ctypes.byref(mw), 0x10, None, 0x20, 0x30, M, 2, dt, 0x40, ws, None)
                    assert rc != L.ERR_WORKSPACE, ("moe", layout, g_idx, K, N, M, dt, lib.q4_last_error())
                    rc = lib.q4_moe_linear_gate_up(ctypes.byref(mw), 0x10, None, 0x20, 0x30, M, 2, dt, 0, 0x40, ws, None)
                    assert rc != L.ERR_WORKSPACE, ("moe fused", layout, g_idx, K, N, M, dt, lib.q4_last_error())


def test_workspace_sizing_other_group_sizes_and_70b_shapes(pkg):
    """Act-order weights with other group sizes than 128 pick other K splits (their parameter
    table shares LDS with the slab): both the per-shape bound and the per-weight size must cover
    what the launcher then asks for."""
    lib = pkg._lib.load()
    L = pkg._lib
    for K, N in [(8192, 28672), (28672, 8192), (8192, 10240), (4096, 4096)]:
        for gs in (32, 64, 128, 256):
            for layout, g_idx in ((0, True), (0, False), (1, False)):
                for M in (1, 2, 4, 8, 12, 16):
                    for dt in (0, 1):
                        w = _weight(pkg, K, N, gs, layout, g_idx)
                        for ws in (lib.q4_workspace_bytes(M, K, N), lib.q4_workspace_bytes_for(ctypes.byref(w), M)):
                            rc = lib.q4_linear(ctypes.byref(w), 0x10, None, 0x20, M, dt, 0x40, ws, None)
                            assert rc != L.ERR_WORKSPACE, (layout, g_idx, K, N, gs, M, dt, lib.q4_last_error())
                        if layout == 0 and not g_idx and N % 128 == 0:
                            ws = lib.q4_workspace_bytes_for(ctypes.byref(w), M)
                            rc = lib.q4_linear_gate_up(ctypes.byref(w), 0x10, None, 0x20, M, dt, 0, 0x40, ws, None)
                            assert rc != L.ERR_WORKSPACE, ("gate_up", K, N, gs, M, dt, lib.q4_last_error())


@pytest.mark.parametrize("K,N,gs,without", [(65536, 24576, 1024, True), (65536, 28672, 1024, True), (65536, 32768, 1024, True), (65536, 57344, 1024, True),
                                            (61440, 49152, 640, True), (81920, 24576, 81920, False), (131072, 28672, 131072, False), (8192, 57344, 128, True)])
def test_gated_act_order_plan_and_launch_agree(pkg, K, N, gs, without):
    """A gated act-order call that the plan says is one launch is not refused for its LDS: with a full workspace never, without one where
    the groups of all K rows fit beside the table of 64 columns."""
    lib, L, fused = pkg._lib.load(), pkg._lib, ctypes.c_int(0)
    for M in (1, 4, 5, 16, 17):
        for dt in (0, 1):
            w = _weight(pkg, K, N, gs, g_idx=True)
            assert lib.q4_linear_gate_up_act_order_plan(ctypes.byref(w), M, dt, ctypes.byref(fused)) == 0 and fused.value == 1
            rc = lib.q4_linear_gate_up_act_order(ctypes.byref(w), 0x10, None, 0x20, M, dt, 0, 0x40, lib.q4_workspace_bytes(M, K, N), None)
            assert rc != L.ERR_WORKSPACE, (M, dt, lib.q4_last_error())
            rc = lib.q4_linear_gate_up_act_order(ctypes.byref(w), 0x10, None, 0x20, M, dt, 0, None, 0, None)
            assert (rc != L.ERR_WORKSPACE) == without, (M, dt, lib.q4_last_error())


def test_linear_plan_matches_its_parts(pkg):
    lib = pkg._lib.load()
    L = pkg._lib
    path, need = ctypes.c_int(0), ctypes.c_size_t(0)
    for layout, g_idx in ((0, False), (0, True), (1, False)):
        for M in (1, 16, 17, 64, 2048):
            w = _weight(pkg, 4096, 6144, 128, layout, g_idx)
            assert lib.q4_linear_plan(ctypes.byref(w), M, 0, ctypes.byref(path), ctypes.byref(need)) == 0
            assert path.value == lib.q4_select_path(ctypes.byref(w), M, 0)
            assert need.value == lib.q4_workspace_bytes_for(ctypes.byref(w), M)
            assert L.WORKSPACE_COUNTER_BYTES <= need.value <= lib.q4_workspace_bytes(M, 4096, 6144)
    w = _weight(pkg, 4096, 6144, 128)
    assert lib.q4_linear_plan(ctypes.byref(w), 1, 0, None, ctypes.byref(need)) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_linear_plan(ctypes.byref(w), 1, 9, ctypes.byref(path), ctypes.byref(need)) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_linear_plan(None, 1, 0, ctypes.byref(path), ctypes.byref(need)) == L.ERR_INVALID_ARGUMENT


def test_noalloc_entry_point_validation_without_gpu(pkg):
    lib = pkg._lib.load()
    L = pkg._lib
    assert lib.q4_linear_noalloc(None, 0x10, None, 0x20, 1, 0, None) == L.ERR_INVALID_ARGUMENT
    w = _weight(pkg, 4096, 4096, 128)
    assert lib.q4_linear_noalloc(ctypes.byref(w), 0x10, None, 0x20, -1, 0, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_linear_noalloc(ctypes.byref(w), 0x10, None, 0x20, 1, 5, None) == L.ERR_INVALID_ARGUMENT
    assert lib.q4_linear_noalloc(ctypes.byref(w), None, None, None, 0, 0, None) == 0  # no rows: nothing to do


@pytest.mark.parametrize("K,N,gs,layout,g_idx,M,dtype,gate_up,want", [
    # decode: one to four fp16 rows keep their own kernels, the gated epilogue and bf16 start at one
    (4096, 6144, 128, 0, False, 1, "f16", 0, "gemv"), (4096, 6144, 128, 0, False, 5, "f16", 0, "batch"),
    (4096, 28672, 128, 0, False, 1, "f16", 1, "batch"), (3584, 37888, 128, 0, False, 13, "bf16", 0, "batch"),
    (4096, 28672, 128, 0, False, 3, "bf16", 0, "gemv"), (8192, 57344, 128, 0, False, 16, "f16", 1, "none"),
    (14336, 4096, 64, 0, False, 1, "f16", 0, "batch"), (4096, 14336, 32, 0, False, 37, "f16", 0, "batch"),
    (4608, 28672, 384, 0, False, 1, "f16", 1, "gemv"), (4096, 6144, 128, 0, False, 64, "f16", 0, "batch"),
    (14336, 4096, 128, 0, False, 49, "f16", 0, "batch"), (14336, 8192, 128, 0, False, 49, "f16", 0, "gemm"),
    (4096, 28672, 128, 1, False, 1, "f16", 0, "gemv"), (4096, 28672, 128, 1, False, 16, "f16", 1, "batch"),
    (4096, 4096, 128, 1, False, 1, "f16", 0, "batch"), (14336, 4096, 128, 1, False, 33, "f16", 0, "gemm"),
    (8192, 10240, 128, 0, True, 4, "f16", 0, "gemv"), (8192, 10240, 128, 0, True, 33, "f16", 0, "batch"),
    (8192, 10240, 128, 0, True, 4, "f16", 1, "batch"), (8192, 10240, 128, 0, True, 6, "f16", 0, "batch"),
    (18944, 3584, 128, 0, True, 2, "bf16", 0, "gemv"), (18944, 3584, 128, 0, True, 3, "bf16", 0, "batch"),
    (8192, 57344, 32, 0, True, 2, "f16", 1, "batch"), (8192, 57344, 32, 0, True, 3, "f16", 1, "none"),
    (8192, 57344, 32, 0, True, 16, "bf16", 0, "gemv"), (8192, 57344, 32, 0, True, 17, "bf16", 0, "batch"),
    (4096, 4096, 128, 0, True, 64, "f16", 1, "batch"), (4096, 4096, 128, 0, True, 65, "f16", 1, "none"),
    (4096, 4096, 128, 0, True, 65, "f16", 0, "gemm"), (4096, 4160, 128, 0, True, 1, "f16", 1, "none"),
    (8192, 57344, 128, 1, False, 5, "f16", 0, "gemv"), (8192, 57344, 128, 1, False, 5, "bf16", 1, "none"),
    (8192, 57344, 128, 1, False, 7, "f16", 0, "batch"), (8192, 57344, 128, 1, False, 7, "f16", 1, "batch"),
    (3584, 37888, 128, 1, False, 32, "f16", 0, "batch"), (3584, 37888, 128, 1, False, 33, "f16", 0, "gemm"),
    (3584, 37888, 128, 0, False, 49, "bf16", 0, "gemm"), (3584, 37888, 128, 0, False, 49, "bf16", 1, "batch"),
    (3584, 37888, 128, 0, False, 49, "f16", 0, "batch"),
    # deals of K over power-of-two splits that come out uneven are left to the older kernels
    (4608, 4608, 32, 0, False, 3, "f16", 0, "gemv"), (4608, 4608, 32, 0, False, 4, "f16", 0, "batch"), (4608, 4608, 32, 0, False, 1, "bf16", 0, "batch"),
    (5760, 8704, 32, 0, False, 48, "f16", 0, "batch"), (5760, 8704, 32, 0, False, 49, "f16", 0, "gemm"), (5760, 8704, 32, 0, False, 49, "f16", 1, "batch"),
    (3584, 37888, 32, 0, False, 64, "bf16", 1, "none"), (2432, 1024, 32, 0, False, 49, "f16", 0, "gemv"),
    (3584, 8192, 128, 1, False, 1, "bf16", 1, "none"), (3584, 8192, 32, 1, False, 1, "bf16", 1, "batch"), (4096, 6144, 128, 1, False, 1, "bf16", 1, "batch"),
    (8192, 10240, 128, 1, False, 4, "bf16", 1, "none"), (4096, 22016, 128, 1, False, 4, "bf16", 1, "batch"), (8192, 10240, 32, 1, False, 4, "f16", 1, "none"),
    (5760, 8704, 128, 1, False, 2, "bf16", 0, "gemv"), (5760, 8704, 128, 1, False, 3, "bf16", 0, "batch"),
    (8192, 10240, 32, 0, True, 16, "f16", 1, "none"), (8192, 10240, 32, 0, True, 17, "f16", 1, "batch"), (8192, 10240, 32, 0, True, 3, "bf16", 1, "batch"),
    # prefill
    (4096, 6144, 128, 0, False, 2048, "bf16", 0, "gemm"), (4096, 28672, 128, 0, False, 2048, "bf16", 1, "gemm"),
    (4096, 28672, 128, 0, False, 301, "f16", 1, "tall"), (14336, 4096, 128, 0, False, 301, "f16", 0, "tall"),
    (4096, 28672, 128, 0, False, 1000, "f16", 1, "block"), (14336, 4096, 128, 1, False, 1000, "f16", 0, "block"),
    (14336, 4096, 128, 1, False, 1000, "bf16", 0, "tall"), (4096, 28672, 32, 0, False, 301, "f16", 0, "gemm"),
    (4096, 28672, 128, 0, False, 2048, "bf16", 0, "gemm"), (4096, 28672, 128, 0, False, 1000, "bf16", 0, "tall"),
    (4096, 12288, 128, 0, False, 2048, "f16", 0, "gemm"), (4096, 12288, 128, 0, False, 2048, "f16", 1, "gemm"),
    (4096, 4096, 128, 0, False, 1400, "f16", 0, "gemm"), (4096, 4096, 128, 0, False, 700, "f16", 0, "tall"),
    (1024, 8192, 128, 1, False, 1000, "f16", 0, "gemm"), (1024, 8192, 128, 1, False, 1000, "f16", 1, "tall"),
    (1024, 8192, 128, 1, False, 512, "bf16", 1, "none"), (1024, 8192, 128, 1, False, 100, "bf16", 0, "tall"),
    (1024, 8192, 128, 1, False, 2048, "f16", 0, "block"), (8192, 57344, 128, 0, False, 2048, "bf16", 0, "tall"),
    (4104, 4104, 8, 0, False, 16, "f16", 0, "generic"), (4104, 4104, 8, 0, False, 16, "f16", 1, "none"),
])
def test_the_kernel_of_a_call(pkg, K, N, gs, layout, g_idx, M, dtype, gate_up, want):
    """Which kernels the library's own choice runs (the sides of the measured crossovers); a forced path runs its own."""
    w = _weight(pkg, K, N, gs, layout, g_idx)
    rc = pkg._lib.load().q4_linear_kernel(ctypes.byref(w), M, 1 if dtype == "bf16" else 0, gate_up)
    assert pkg._lib.KERNEL_NAMES[rc] == want


def _all_tiles(pkg, M, K, N, gs, dtype, layout=0, gate_up=0, g_idx=False):
    """(rows, columns, K parts inside a workgroup, workgroups along K)"""
    out, w = (ctypes.c_int * 4)(-1, -1, -1, -1), _weight(pkg, K, N, gs, layout, g_idx)
    assert pkg._lib.load().q4_linear_tiles(ctypes.byref(w), M, 1 if dtype == "bf16" else 0, gate_up, out) == 0
    return tuple(out)


def _tiles(pkg, M, K, N, gs, dtype, **kw):
    """Of a prefill call: (rows, workgroups along K, K halves)"""
    rows, columns, halves, splits = _all_tiles(pkg, M, K, N, gs, dtype, **kw)
    assert columns * halves == (256 if rows else 0)
    return rows, splits, halves


def test_the_tiles_of_a_prefill_call(pkg):
    """The calls that the GPU test of two K halves means run on two K halves; calls of other kernels have no tiles."""
    from tests.test_tall_gpu import HALVES

    for M, K, N, gs, dtype, rows, splits in HALVES:
        assert _tiles(pkg, M, K, N, gs, dtype) == (rows, splits, 2), (M, K, N)
    # (halves that would go out in two rounds of workgroups over a short K)
    assert _tiles(pkg, 167, 1024, 16640, 128, "f16") == (96, 1, 1) and _tiles(pkg, 794, 1152, 17664, 128, "f16")[2] == 1
    assert _tiles(pkg, 638, 896, 18944, 128, "f16") == (256, 1, 1) and _tiles(pkg, 258, 5632, 45056, 128, "bf16")[2] == 2
    # (160-row tiles whose halves are four or five K tiles)
    assert _tiles(pkg, 825, 640, 4864, 128, "f16") == (96, 1, 1) and _tiles(pkg, 679, 512, 6144, 128, "f16") == (96, 1, 1)
    # (halves on 96-row tiles beyond 1024 rows, where whole K ranges on such tiles are left out)
    for K, N, M in ((5120, 2304, 1025), (5504, 2304, 1025), (4864, 2304, 1099), (4864, 2048, 1173), (4864, 1792, 1432), (4096, 2048, 1245)):
        assert _tiles(pkg, M, K, N, 128, "f16") == (96, 1, 2)
    # (tiles that are a third padding)
    assert _tiles(pkg, 104, 4096, 4096, 128, "f16") == (96, 4, 2) and _tiles(pkg, 203, 4096, 12288, 128, "f16") == (128, 1, 2)
    assert _tiles(pkg, 161, 8192, 8192, 128, "f16") == (96, 4, 1) and _tiles(pkg, 1000, 4096, 28672, 128, "f16", gate_up=1) == (256, 1, 1)
    assert _tiles(pkg, 2048, 4096, 28672, 128, "bf16") == (0, 0, 0) and _tiles(pkg, 301, 4104, 4104, 8, "f16") == (0, 0, 0)
    w = _weight(pkg, 4096, 4096, 128)
    assert pkg._lib.load().q4_linear_tiles(ctypes.byref(w), 301, 0, 0, None) == pkg._lib.ERR_INVALID_ARGUMENT


def _launched(pkg, w, M, dtype, gate_up=0, path=0):
    """The launch that a call with a full workspace ends at (it fails for want of a GPU, and says its name), or the error code."""
    lib = pkg._lib.load()
    ws = lib.q4_workspace_bytes(M, w.K, w.N)
    if gate_up:
        rc = lib.q4_linear_gate_up(ctypes.byref(w), 0x10, None, 0x20, M, dtype, 0, 0x40, ws, None)
    else:
        rc = lib.q4_linear_ex(ctypes.byref(w), 0x10, None, 0x20, M, dtype, 0x40, ws, path, None)
    return lib.q4_last_error().decode().split(":")[0] if rc == pkg._lib.ERR_LAUNCH else rc


@pytest.mark.parametrize("M,K,N,gs,gate_up,want", [(5, 13312, 27392, 64, 0, 8), (31, 3584, 28672, 64, 0, 8), (10, 3968, 28672, 64, 0, 8), (2, 3072, 24960, 64, 0, 8),
                                                  (1, 4096, 28672, 128, 1, 4), (31, 8192, 28672, 128, 0, 4), (5, 4096, 28672, 32, 0, 8)])
def test_k_waves_of_unsplit_batch_tiles(pkg, M, K, N, gs, gate_up, want):
    """Four waves for 128-column tiles that fill the chip, eight in groups of 64 and 32 rows."""
    assert _all_tiles(pkg, M, K, N, gs, "f16", gate_up=gate_up) == ((M + 15) // 16 * 16, 128, want, 1)


@pytest.mark.parametrize("M,K,N,gs,dtype,gate_up,want", [(8, 2560, 10112, 64, "f16", 0, (16, 64, 8, 1)), (5, 12800, 18816, 64, "bf16", 1, (16, 64, 8, 2)),
                                                        (11, 8704, 3584, 128, "f16", 0, (16, 64, 8, 4)), (13, 2304, 50816, 128, "f16", 1, (16, 64, 4, 1)),
                                                        (4, 8192, 57344, 128, "f16", 1, (16, 128, 4, 4)), (4, 4096, 28672, 128, "f16", 1, (16, 128, 8, 1)), (39, 18688, 10624, 128, "bf16", 1, (48, 64, 4, 3)), (48, 13440, 2304, 128, "bf16", 0, (48, 64, 8, 7))])
def test_splits_of_the_act_order_batch_kernel(pkg, M, K, N, gs, dtype, gate_up, want):
    """Powers of two unless another number is well ahead of them, eight waves kept at more than that."""
    assert _all_tiles(pkg, M, K, N, gs, dtype, gate_up=gate_up, g_idx=True) == want


FEW = "q4_linear(AWQ, up to four rows)"


@pytest.mark.parametrize("K,N,layout,g_idx,M,dtype,kernel,tiles", [
    (4096, 28672, 1, False, 1, "f16", FEW, (4, 256, 8, 2)), (14336, 4096, 1, False, 4, "bf16", FEW, (4, 256, 8, 14)),
    (8192, 57344, 1, False, 5, "f16", "q4_linear(AWQ, five to sixteen rows)", (16, 256, 8, 1)),
    (8192, 10240, 0, True, 4, "f16", "q4_linear(act-order batch kernel)", (16, 64, 8, 3))])
def test_a_forced_decode_path_runs_its_own_kernels(pkg, K, N, layout, g_idx, M, dtype, kernel, tiles):
    """Decode calls that are named for their path and run on a batch kernel's variant: only where the caller leaves the choice, and only with
    the workspace that the path asks for."""
    lib, L, dt = pkg._lib.load(), pkg._lib, 1 if dtype == "bf16" else 0
    w = _weight(pkg, K, N, 128, layout, g_idx)
    assert _launched(pkg, w, M, dt) == kernel and _all_tiles(pkg, M, K, N, 128, dtype, layout=layout, g_idx=g_idx) == tiles
    assert _launched(pkg, w, M, dt, path=L.PATH_GEMV) == "q4_linear(gemv)"
    if L.KERNEL_NAMES[lib.q4_linear_kernel(ctypes.byref(w), M, dt, 0)] == "gemv":
        lib.q4_linear_ex(ctypes.byref(w), 0x10, None, 0x20, M, dt, 0x40, L.WORKSPACE_COUNTER_BYTES - 16, L.PATH_AUTO, None)
        assert kernel.encode() not in lib.q4_last_error()


# (K in whole 128-row chunks, one and more a wave; fewer and more units of 128 x 256 weights than the chip has SIMDs)
@pytest.mark.parametrize("K,N,gate_up,dtype,few", [(2176, 4096, 0, 0, False), (2176, 16384, 0, 0, True), (2176, 8960, 0, 0, False), (2176, 9216, 0, 0, True), (3968, 8192, 0, 1, False), (2048, 512, 0, 0, True), (8320, 1024, 0, 1, True),
                                                   (2176, 4096, 1, 0, False), (2176, 20480, 1, 0, True), (11008, 2048, 1, 0, False), (11008, 3072, 1, 0, True),
                                                   (2048, 4096, 1, 0, True), (4096, 4096, 1, 1, False), (4096, 8192, 1, 1, True)])
def test_awq_rows_of_small_ragged_layers(pkg, K, N, gate_up, dtype, few):
    for M in (1, 4):
        got = _launched(pkg, _weight(pkg, K, N, 128, layout=1), M, dtype, gate_up)
        assert (got == FEW) == few, (M, got)


@pytest.mark.parametrize("K,N,gs,M,want", [(8192, 32768, 128, 33, 0), (8192, 32768, 128, 64, 0), (8192, 57344, 32, 48, 0), (8256, 33024, 64, 32, 0),
                                          (8256, 33024, 64, 33, 1), (8256, 57344, 64, 64, 1), (8256, 57344, 64, 65, 0), (8256, 28672, 64, 48, 0),
                                          (8192, 32768, 128, 128, 0), (8192, 32768, 128, 129, 1)])
def test_decode_batches_regroup_where_no_kernel_reads_through_g_idx(pkg, K, N, gs, M, want):
    """33-64 rows: the act-order batch kernel's calls are never regrouped, the widest of the others are."""
    lib, w = pkg._lib.load(), _weight(pkg, K, N, gs, g_idx=True)
    need, scratch = ctypes.c_size_t(0), ctypes.c_size_t(0)
    for dtype in (0, 1):
        assert lib.q4_linear_regroup_plan(ctypes.byref(w), M, dtype, 0, ctypes.byref(need), ctypes.byref(scratch)) == want
        assert not (want and pkg._lib.KERNEL_NAMES[lib.q4_linear_kernel(ctypes.byref(w), M, dtype, 0)] == "batch")


@pytest.mark.parametrize("E,topk,K,N,tokens,gate_up,want", [
    (8, 2, 4096, 28672, 192, 1, "batch"), (8, 2, 14336, 4096, 192, 0, "batch"), (8, 2, 14336, 4096, 193, 0, "gemm"),
    (64, 6, 1408, 2048, 48, 0, "batch"), (64, 6, 1408, 2048, 64, 0, "gemv"), (64, 6, 1408, 2048, 192, 0, "gemm"),
    (64, 6, 2048, 2816, 170, 1, "batch"), (64, 6, 2048, 2816, 192, 1, "none"),
    (16, 4, 4096, 2048, 64, 0, "batch"), (16, 4, 4096, 2048, 128, 0, "gemm"), (16, 4, 2048, 8192, 192, 1, "batch"),
])
def test_the_kernel_of_a_grouped_call(pkg, E, topk, K, N, tokens, gate_up, want):
    lib, L = pkg._lib.load(), pkg._lib
    w = L.Q4MoeWeight(_weight(pkg, K, N, 128), E, K * N // 8, K * N // 1024, K * N // 128, 0)
    for dtype in (0, 1):
        assert L.KERNEL_NAMES[lib.q4_moe_kernel(ctypes.byref(w), tokens, topk, dtype, gate_up)] == want


def test_path_selection_and_workspace(pkg):
    lib = pkg._lib.load()
    L = pkg._lib
    w = _weight(pkg, 4096, 4096, 128)
    for M, want in [(1, L.PATH_GEMV), (16, L.PATH_GEMV), (64, L.PATH_GEMV), (65, L.PATH_GEMM), (2048, L.PATH_GEMM)]:
        assert lib.q4_select_path(ctypes.byref(w), M, 0) == want
    # the decode kernel's reach depends on the shape (measured crossovers); 17..20 rows stay on it
    # while the activation slab of the 16-row configuration still fits LDS
    for K, N, last_gemv in [(4096, 6144, 32), (4096, 14336, 32), (4096, 28672, 18), (8192, 8192, 20), (8192, 10240, 18), (14336, 4096, 20), (6144, 6144, 20)]:
        w2 = _weight(pkg, K, N, 128)
        assert lib.q4_select_path(ctypes.byref(w2), last_gemv, 0) == L.PATH_GEMV, (K, N)
        assert lib.q4_select_path(ctypes.byref(w2), last_gemv + 1, 0) == L.PATH_GEMM, (K, N)
    assert int(dict(re.findall(r"#define\s+(Q4_KERNEL_[A-Z]+)\s+(\d+)", HEADER.read_text()))["Q4_KERNEL_BATCH"]) == L.KERNEL_BATCH
    odd = _weight(pkg, 4104, 4104, 8)
    assert lib.q4_select_path(ctypes.byref(odd), 1, 0) == L.PATH_GENERIC
    assert lib.q4_select_path(ctypes.byref(odd), 512, 0) == L.PATH_GENERIC
    for M, K, N in [(1, 4096, 4096), (16, 4096, 28672), (16, 14336, 4096), (4, 8192, 10240)]:
        nbytes = lib.q4_workspace_bytes(M, K, N)
        assert nbytes >= L.WORKSPACE_COUNTER_BYTES + M * N * 4
        assert nbytes <= L.WORKSPACE_COUNTER_BYTES + 64 * 16 * N * 4
    assert lib.q4_workspace_bytes(0, 0, 0) == L.WORKSPACE_COUNTER_BYTES


def _cpu_gptq_tensors(oracle, K=256, N=64, gs=128, **kw):
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=0, **kw)
    t = lambda a: None if a is None else torch.from_numpy(a)
    return t(qw), t(qz), t(sc), t(gi)


def test_gptq_weight_contract(pkg, oracle):
    qw, qz, sc, _ = _cpu_gptq_tensors(oracle)
    w = pkg.GPTQWeight(qw, qz, sc.float(), None, 4, 128, use_awq_kernel=False, use_exllama=False)
    assert w.scales.dtype == torch.float16        # fp32 scales are narrowed (gptq/__init__.py:29-31)
    assert w.device == qw.device
    lin = pkg.get_linear(w, None)
    assert type(lin).__name__ == "QuantLinear"
    assert (lin.infeatures, lin.outfeatures, lin.bits, lin.maxq, lin.groupsize) == (256, 64, 4, 15, 128)
    assert lin.bias is None
    ex = pkg.get_linear(pkg.GPTQWeight(qw, qz, sc, None, 4, 128, False, True), torch.zeros(64, dtype=torch.float16))
    assert type(ex).__name__ == "ExllamaQuantLinear" and ex.infeatures == 256 and ex.outfeatures == 64
    assert ex.act_order is False
    with pytest.raises(NotImplementedError):
        pkg.get_linear(torch.zeros(2, 2), None)


def test_bits_other_than_four_are_rejected(pkg, oracle):
    qw, qz, sc, _ = _cpu_gptq_tensors(oracle)
    with pytest.raises(NotImplementedError, match="4 bits"):
        pkg.QuantLinear(qw, qz, sc, None, None, 8, 128)
    with pytest.raises(NotImplementedError):
        pkg.QuantLinear.new(2, 128, 256, 64, False)
    with pytest.raises(ValueError, match="bits=4"):
        pkg.ExllamaQuantLinear(pkg.GPTQWeight(qw, qz, sc, None, 8, 128, False, True), None)
    with pytest.raises(NotImplementedError, match="4-bit"):
        pkg.WQLinear(8, 128, qw, qz, sc, None)
    # bits read from a marker tensor arrive as a float (tests/utils/test_weights.py:671-672)
    assert pkg.QuantLinear(qw, qz, sc, None, None, 4.0, 128).bits == 4


def test_quant_linear_new_geometry(pkg):
    lin = pkg.QuantLinear.new(4, 128, 1024, 512, True)
    assert lin.qweight.shape == (128, 512) and lin.qweight.dtype == torch.int32
    assert lin.qzeros.shape == (8, 64) and lin.scales.shape == (8, 512)
    assert lin.g_idx.tolist() == [i // 128 for i in range(1024)]
    assert lin.bias.shape == (512,) and lin.bias.dtype == torch.float16
    one_group = pkg.QuantLinear.new(4, -1, 1024, 512, False)
    assert one_group.qzeros.shape == (1, 64) and one_group.bias is None


def test_wqlinear_contract(pkg, oracle):
    aq, az, sc = oracle.make_awq(256, 64, 128, seed=0)
    lin = pkg.WQLinear(4, 128, torch.from_numpy(aq), torch.from_numpy(az), torch.from_numpy(sc), None)
    assert (lin.in_features, lin.out_features, lin.w_bit, lin.group_size) == (256, 64, 4, 128)
    assert pkg.WQLinear(4, -1, torch.from_numpy(aq), torch.from_numpy(az[:1]), torch.from_numpy(sc[:1]), None).group_size == 256
    with pytest.raises(AssertionError):
        pkg.WQLinear(4, 96, torch.from_numpy(aq), torch.from_numpy(az), torch.from_numpy(sc), None)
    w = pkg.GPTQWeight(torch.from_numpy(aq), torch.from_numpy(az), torch.from_numpy(sc), None, 4, 128, True, False)
    assert type(pkg.get_linear(w, None)).__name__ == "WQLinear"  # no ROCm refusal here


def test_no_cpu_fallback(pkg, oracle):
    """CPU tensors are refused loudly: the package has no host compute path."""
    qw, qz, sc, _ = _cpu_gptq_tensors(oracle)
    lin = pkg.QuantLinear(qw, qz, sc, None, None, 4, 128)
    with pytest.raises(RuntimeError, match="GPU only"):
        lin(torch.zeros(1, 256, dtype=torch.float16))
    with pytest.raises(RuntimeError, match="GPU only"):
        lin.dequantize()


@pytest.mark.parametrize("layout,g_idx", [(0, False), (0, True), (1, False)])
def test_weights_on_another_gpu_are_refused(pkg, monkeypatch, layout, g_idx):
    """Nothing is launched with the addresses of two GPUs (stand-ins for the tensors: there are no two here)."""
    from types import SimpleNamespace

    at = lambda i, **kw: SimpleNamespace(is_cuda=True, device=torch.device("cuda", i), data_ptr=lambda: 0x1000, **kw)  # noqa: E731
    x = at(1, dtype=torch.float16, shape=(4, 4096), dim=lambda: 2, is_contiguous=lambda: True)
    w = pkg.ops.PackedWeight(at(0), at(0), at(0), at(0) if g_idx else None, 4096, 8192, 128, 32, layout)
    monkeypatch.setattr(pkg.ops, "_launch_linear", lambda *a: pytest.fail("launched"))
    for call in (pkg.ops.linear, pkg.ops.linear_gate_up):
        with pytest.raises(RuntimeError, match="weights on cuda:0"):
            call(w, x)


@pytest.mark.parametrize("why", ["missing", "built against torch"])
def test_calls_without_the_extension_module(pkg, oracle, monkeypatch, tmp_path, why):
    """The Python code answers where the eager call's module cannot be used; without the library nothing does."""
    qw, qz, sc, _ = _cpu_gptq_tensors(oracle)
    pk = pkg.ops.make_packed(qw, qz, sc, None, 128, 0)
    monkeypatch.setattr(pkg._lib, "_call", None)
    if why == "missing":
        monkeypatch.setattr(pkg._lib, "CALL_PATH", tmp_path / "_q4call.so")
    else:
        monkeypatch.setattr(torch, "__version__", "2.0.0")
    with pytest.warns(RuntimeWarning, match=why):
        call = pk.call()
    x = torch.zeros(1, 256, dtype=torch.float16)
    assert call(x, None) is None and call(x, None, pk) is None
    with pytest.raises(RuntimeError, match="GPU only"):  # linear's own answer to a tensor on the CPU
        pkg.ops.apply_linear(pk, x, None)
    monkeypatch.setattr(pkg._lib, "_lib", None)
    monkeypatch.setattr(pkg._lib, "LIB_PATH", tmp_path / "libq4linear.so")
    monkeypatch.setattr(pkg._lib, "_call", None)
    with pytest.raises(ImportError, match="no fallback"):
        pkg.ops.make_packed(qw, qz, sc, None, 128, 0).call()


def test_nested_activations_raise(pkg, oracle):
    """Tensors whose sizes throw come back as a Python error (in a process of their own: what a C++ exception ends is the process)."""
    import subprocess
    import sys

    code = (
        "import importlib, torch, warnings; warnings.simplefilter('ignore')\n"
        "pkg = importlib.import_module('text-generation-inference_amd')\n"
        "i = lambda *s: torch.zeros(s, dtype=torch.int32)\n"
        "pk = pkg.ops.make_packed(i(32, 64), i(2, 8), torch.ones(2, 64, dtype=torch.float16), None, 128, 0)\n"
        "x = torch.nested.nested_tensor([torch.zeros(2, 256), torch.zeros(3, 200)], dtype=torch.float16)\n"
        "try:\n    pkg.ops.apply_linear(pk, x, None)\nexcept RuntimeError:\n    print('raised')\n"
    )
    got = subprocess.run([sys.executable, "-c", code], cwd=HEADER.parent.parent, capture_output=True, text=True, timeout=300)
    assert got.returncode == 0 and got.stdout.strip() == "raised", got.stderr[-2000:]


def test_make_packed_validation(pkg, oracle):
    qw, qz, sc, gi = _cpu_gptq_tensors(oracle, act_order=True)
    mk = pkg.ops.make_packed
    pk = mk(qw, qz, sc, gi, 128, 0)
    assert (pk.K, pk.N, pk.groupsize, pk.num_groups) == (256, 64, 128, 2)
    assert mk(qw, qz[:1], sc[:1], None, -1, 0).groupsize == 256
    with pytest.raises(TypeError):
        mk(qw.to(torch.int64), qz, sc, None, 128, 0)
    with pytest.raises(TypeError):
        mk(qw, qz, sc.float(), None, 128, 0)
    with pytest.raises(ValueError, match="inconsistent"):
        mk(qw, qz[:, :4], sc, None, 128, 0)
    with pytest.raises(ValueError, match="do not cover"):
        mk(qw, qz[:1], sc[:1], None, 128, 0)
    with pytest.raises(ValueError, match="g_idx has"):
        mk(qw, qz, sc, gi[:100], 128, 0)
    with pytest.raises(ValueError, match="AWQ"):
        mk(torch.zeros(256, 8, dtype=torch.int32), qz, sc, gi, 128, 1)


def test_trivial_g_idx_detection(pkg):
    from importlib import import_module
    ql = import_module("text-generation-inference_amd.layers.gptq.quant_linear")
    seq = (torch.arange(512) // 128).to(torch.int32)
    assert ql.is_trivial_g_idx(seq, 128)
    assert ql.is_trivial_g_idx(torch.zeros(512, dtype=torch.int32), -1)
    assert not ql.is_trivial_g_idx(seq.flip(0), 128)
    assert not ql.is_trivial_g_idx(seq, 64)


def test_conversion_utils_match_oracle(pkg, oracle):
    """The torch layout helpers (loader-side host logic) agree with the oracle's NumPy ones."""
    cu = pkg.conversion_utils
    aq, az, sc = oracle.make_awq(128, 64, 32, seed=3)
    gq, gz = cu.fast_awq_to_gptq(torch.from_numpy(aq), torch.from_numpy(az))
    oq, oz = oracle.fast_awq_to_gptq(aq, az)
    assert np.array_equal(gq.numpy(), oq) and np.array_equal(gz.numpy(), oz)
    m = torch.randint(0, 16, (32, 64), generator=torch.Generator().manual_seed(0))
    for d in ("row", "column"):
        assert torch.equal(cu.unpack(cu.pack(m, d), d).to(torch.int64), m)
    assert np.array_equal(cu.pack(m, "row").numpy(), oracle.pack_rows(m.numpy()))
    assert np.array_equal(cu.pack(m, "column").numpy(), oracle.pack_cols(m.numpy()))
    assert cu.AWQ_PACK_ORDER == oracle.AWQ_PACK_ORDER


def test_exllama_hooks_are_noops(pkg):
    pkg.set_device(torch.device("cpu"))
    assert pkg.create_exllama_buffers(4096) is None


def test_misaligned_pointers_are_refused(pkg):
    """The kernels fetch with 16-byte loads: tensors, activations, outputs and workspaces off a
    16-byte boundary are turned away before anything is launched (fake pointers, never read)."""
    L = pkg._lib
    lib = L.load()
    good = _weight(pkg, 4096, 4096, 128)
    for field in ("qweight", "qzeros", "scales"):
        w = _weight(pkg, 4096, 4096, 128)
        setattr(w, field, getattr(w, field) + 4)
        assert lib.q4_linear(ctypes.byref(w), 0x100, None, 0x200, 1, 0, 0x400, 1 << 20, None) == L.ERR_INVALID_ARGUMENT
        assert b"aligned" in lib.q4_last_error()
    w = _weight(pkg, 4096, 4096, 128, g_idx=True)
    w.g_idx = w.g_idx + 8
    assert lib.q4_linear(ctypes.byref(w), 0x100, None, 0x200, 1, 0, 0x400, 1 << 20, None) == L.ERR_INVALID_ARGUMENT
    for x, bias, y, ws in [(0x102, None, 0x200, 0x400), (0x100, None, 0x208, 0x400), (0x100, 0x301, 0x200, 0x400),
                           (0x100, None, 0x200, 0x404)]:
        assert lib.q4_linear(ctypes.byref(good), x, bias, y, 1, 0, ws, 1 << 20, None) == L.ERR_INVALID_ARGUMENT
        assert b"aligned" in lib.q4_last_error()
