"""Prefill kernels with tiles that follow M (q4_gemm_tall.cuh, q4_gemm_block.cuh) at the edges of their row
tiles, K tiles and splits, against the oracle.

Bars as in the other parity tests: max|y - ref| / max|ref| <= 2e-3 in fp16 (output rounding 2^-11 plus
the fp32 accumulation), 8e-3 in bf16 (output rounding 2^-8); the gated epilogue has three roundings of
that size and the same bars, as in test_gate_up_gpu.py.
"""

import ctypes

import numpy as np
import pytest
import torch

from tests.util import max_rel_err, to_dev, to_f32

pytestmark = pytest.mark.gpu

TOL = {"f16": 2e-3, "bf16": 8e-3}


def _weight(pkg, oracle, gpu, layout, K, N, g, seed, dtype):
    if layout == "awq":
        qw, qz, sc = oracle.make_awq(K, N, g, seed=seed)
        return pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 1), oracle.dequant_awq(qw, qz, sc, g, dtype)
    qw, qz, sc, _ = oracle.make_gptq(K, N, g, seed=seed, sym=False)
    return pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 0), oracle.dequant_gptq(qw, qz, sc, None, g, dtype)


# On 112 column tiles the row counts 65, 225, 301, 420 and 700 are tiled in 96, 128, 160, 256 and 192 rows (one row more
# than a tile, ragged and full ones); K in one, two, three .. seven K tiles of 64 rows (the loop takes four at a time)
@pytest.mark.parametrize("layout", ["gptq", "awq"])
@pytest.mark.parametrize("M,K,dtype", [(65, 64, "f16"), (97, 128, "bf16"), (225, 192, "f16"), (225, 320, "bf16"), (301, 64, "bf16"),
                                       (301, 256, "f16"), (320, 384, "bf16"), (420, 320, "f16"), (420, 128, "bf16"), (512, 448, "f16"),
                                       (700, 64, "f16"), (700, 192, "bf16")])
def test_row_tiles(pkg, oracle, gpu, layout, M, K, dtype):
    N = 28672
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, 64, K + M, dtype)
    bf = dtype == "bf16"
    dt = torch.bfloat16 if bf else torch.float16
    assert all(pkg.ops.kernel_of(pk, M, dt, gate_up) in ("tall", "block") for gate_up in (False, True))
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    b32 = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias = oracle.f32_to_bf16_bits(b32) if bf else b32.astype(np.float16)
    y32, _ = oracle.linear_forward(x, w, bias, dtype)
    got = pkg.ops.linear(pk, to_dev(x, gpu, bf16=bf), to_dev(bias, gpu, bf16=bf))
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]
    _, want = oracle.gate_up_forward(x, w, "silu", bias, dtype)
    got = pkg.ops.linear_gate_up(pk, to_dev(x, gpu, bf16=bf), "silu", to_dev(bias, gpu, bf16=bf))
    assert max_rel_err(to_f32(got), oracle.to_f32(want, dtype)) <= TOL[dtype]


# few column tiles: K splits, ragged over the K tiles (4096 / 64 = 64, 5504 / 64 = 86 in 3, 6, 8)
@pytest.mark.parametrize("layout", ["gptq", "awq"])
@pytest.mark.parametrize("M,K,N,gs,dtype", [(66, 5504, 256, 128, "f16"), (160, 4096, 512, 4096, "bf16"), (257, 5504, 1024, 128, "bf16"),
                                            (301, 5504, 2048, 64, "f16"), (1000, 4096, 1024, 256, "f16"), (1000, 5504, 2048, 128, "bf16")])
def test_splits(pkg, oracle, gpu, layout, M, K, N, gs, dtype):
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, gs, K + M, dtype)
    bf = dtype == "bf16"
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    y32, _ = oracle.linear_forward(x, w, None, dtype)
    xt = to_dev(x, gpu, bf16=bf)
    got = pkg.ops.linear(pk, xt)
    again = pkg.ops.linear(pk, xt)
    assert torch.equal(got, again)
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]


# ... and where the library picks these kernels for them, the 256 x 256 one included; K in 32 and 86 K tiles
@pytest.mark.parametrize("layout,M,K,N,gs,dtype", [
    ("gptq", 66, 2048, 256, 128, "f16"), ("gptq", 700, 4096, 1024, 256, "f16"), ("gptq", 301, 5504, 2048, 128, "bf16"),
    ("gptq", 1000, 2048, 512, 2048, "bf16"), ("awq", 66, 2048, 256, 128, "f16"), ("awq", 301, 5504, 4096, 64, "f16"),
    ("awq", 1000, 5504, 4096, 128, "f16"), ("awq", 512, 5504, 2048, 64, "bf16"), ("awq", 100, 2048, 512, 2048, "bf16")])
def test_splits_of_the_picked_kernels(pkg, oracle, gpu, layout, M, K, N, gs, dtype):
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, gs, K + M, dtype)
    bf = dtype == "bf16"
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16 if bf else torch.float16) in ("tall", "block")
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    y32, _ = oracle.linear_forward(x, w, None, dtype)
    xt = to_dev(x, gpu, bf16=bf)
    got = pkg.ops.linear(pk, xt)
    assert torch.equal(got, pkg.ops.linear(pk, xt))
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]


# GPTQ, two halves of K in a workgroup: 96-, 128- and 160-row tiles, ragged and full, without and with splits in both data types, four K tiles
# a half (1024 x 8192) and more, groups of 64 and one group.  (M, K, N, groupsize, dtype, rows of a tile, splits)
HALVES = [(77, 14336, 4096, 128, "f16", 96, 8), (96, 3584, 8192, 64, "f16", 96, 4), (301, 1024, 8192, 1024, "f16", 96, 1), (301, 1024, 8192, 64, "bf16", 96, 1),
          (420, 1024, 8192, 128, "f16", 128, 1), (85, 4096, 4096, 128, "bf16", 96, 8), (300, 2048, 2048, 64, "f16", 96, 4), (640, 3584, 8192, 128, "f16", 160, 1),
          (96, 4096, 4096, 128, "bf16", 96, 4), (147, 4608, 5632, 128, "f16", 160, 4), (120, 2688, 7168, 128, "bf16", 128, 3), (1245, 4096, 2048, 128, "bf16", 96, 1)]


@pytest.mark.parametrize("M,K,N,gs,dtype", [case[:5] for case in HALVES])
def test_two_halves_of_k(pkg, oracle, gpu, M, K, N, gs, dtype):
    pk, w = _weight(pkg, oracle, gpu, "gptq", K, N, gs, K + M, dtype)
    bf = dtype == "bf16"
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16 if bf else torch.float16) == "tall"
    tiles = (ctypes.c_int * 4)()
    assert pkg._lib.load().q4_linear_tiles(ctypes.byref(pk.struct()), M, int(bf), 0, tiles) == 0 and tiles[2] == 2
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    b32 = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias = oracle.f32_to_bf16_bits(b32) if bf else b32.astype(np.float16)
    y32, _ = oracle.linear_forward(x, w, bias, dtype)
    xt, bt = to_dev(x, gpu, bf16=bf), to_dev(bias, gpu, bf16=bf)
    got = pkg.ops.linear(pk, xt, bt)
    assert torch.equal(got, pkg.ops.linear(pk, xt, bt))
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]
    clean = got.clone()
    xt[3, K // 2], xt[M - 1, 5] = float("inf"), float("nan")
    got = pkg.ops.linear(pk, xt, bt)
    keep = [r for r in range(M) if r not in (3, M - 1)]
    assert torch.equal(got[keep], clean[keep]) and bool(torch.isnan(got[M - 1]).all()) and not bool(torch.isfinite(got[3]).any())


@pytest.mark.parametrize("layout", ["gptq", "awq"])
def test_non_finite_rows_stay_alone(pkg, oracle, gpu, layout):
    """An infinite or undefined activation changes its own row only, the last row of a ragged tile included."""
    M, K, N = 301, 256, 28672
    pk, _ = _weight(pkg, oracle, gpu, layout, K, N, 128, 3, "f16")
    x = oracle.make_x(M, K, seed=8)
    clean = pkg.ops.linear(pk, to_dev(x, gpu)).cpu().numpy()
    x[7, K // 2] = np.inf
    x[300, 5] = np.nan
    got = pkg.ops.linear(pk, to_dev(x, gpu)).cpu().numpy()
    assert np.isnan(got[300]).all() and not np.isfinite(got[7]).any()
    keep = [r for r in range(M) if r not in (7, 300)]
    assert np.array_equal(got[keep], clean[keep])
