"""AWQ decode kernel for five to sixteen rows (q4_gemv_awq_wide.cuh) at the edges of its rows, tiles, K deals and exchange levels.

Bars: the sums are those of x (q - z), scaled, in fp32; an output is off by its own rounding (2^-11 of it in fp16, 2^-8 in bf16) and by
fp32 sums, of which a chunk's 128 terms, K / 128 chunks and at most eight waves and four levels follow each other: 140 + K / 128
roundings of 2^-24 of the sum of the terms' magnitudes.  Gated: three roundings follow each other (sums, activation, product).
"""

import numpy as np
import pytest
import torch

from tests.util import to_dev

pytestmark = pytest.mark.gpu

DT = {"f16": torch.float16, "bf16": torch.bfloat16}
U = {"f16": 2.0**-11, "bf16": 2.0**-8}


def _case(pkg, oracle, gpu, K, N, gs, seed):
    g = K if gs == -1 else gs
    qw, qz, sc = oracle.make_awq(K, N, g, seed=seed)
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 1)
    ints = torch.from_numpy(oracle.dequant_awq(qw, qz, np.ones_like(sc), g, "f16")).to(gpu).double()
    return pk, ints * to_dev(sc, gpu).double().repeat_interleave(g, dim=0)


def _rand(gpu, dtype, seed, *shape):
    return torch.randn(shape, device=gpu, generator=torch.Generator(device=gpu).manual_seed(seed)).to(DT[dtype])


# K: ragged deals (17, 33, 67, 112 chunks), odd numbers of workgroups along K; N: an odd number of tiles, more tiles than CUs
@pytest.mark.parametrize("K,N,gs", [(2176, 24064, 128), (4224, 12544, -1), (8576, 9472, 128), (14336, 4096, 512), (1024, 81920, 256)])
def test_plain(pkg, oracle, gpu, K, N, gs):
    pk, w = _case(pkg, oracle, gpu, K, N, gs, K)
    for M, dtype in [(5, "f16"), (8, "bf16"), (11, "f16"), (16, "f16"), (16, "bf16")]:
        assert pkg.ops.kernel_of(pk, M, DT[dtype]) == "batch"
        x, bias = _rand(gpu, dtype, M, M, K), _rand(gpu, dtype, N, N)
        got = pkg.ops.linear(pk, x)
        assert all(torch.equal(got, pkg.ops.linear(pk, x)) for _ in range(3))  # cells left at zero, no order of arrival in the sums
        want, terms = x.double() @ w, x.double().abs() @ w.abs()
        assert bool(((got.double() - want).abs() <= U[dtype] * want.abs() + (140 + K // 128) * 2.0**-24 * terms + 2.0**-25).all())
        assert torch.equal(pkg.ops.linear(pk, x, bias), got + bias)
        # an infinity, a NaN and a row of zeros under other rows
        x[0, K // 2], x[M - 1, 5], x[2] = float("inf"), float("nan"), 0
        bad = pkg.ops.linear(pk, x)
        wcol = w[K // 2]
        assert bool(torch.where(wcol == 0, torch.isnan(bad[0]), bad[0].float() == torch.sign(wcol).float() * float("inf")).all())
        assert bool(torch.isnan(bad[M - 1]).all()) and not bool(bad[2].view(torch.int16).any())
        assert torch.equal(bad[3 : M - 1], got[3 : M - 1])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_large_activation_under_zero_weights(pkg, oracle, gpu, dtype):
    """Nothing of it reaches the sums: the zero point leaves the weights before they meet x."""
    K, N = 8192, 10240
    qw, qz, sc = oracle.make_awq(K, N, 128, seed=3)
    q, z = oracle.awq_unpack_cols(qw), oracle.awq_unpack_cols(qz)
    q[300] = z[300 // 128]
    pk = pkg.ops.make_packed(to_dev(oracle.awq_pack_cols(q), gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, 128, 1)
    x = _rand(gpu, dtype, 1, 7, K)
    x[1, 300] = 0
    clean = pkg.ops.linear(pk, x)
    x[1, 300] = 6e4 if dtype == "f16" else 2.0**100
    assert torch.equal(pkg.ops.linear(pk, x), clean)


# 46 and 23 pairs of tiles, splits of one (more tiles than CUs) and many
@pytest.mark.parametrize("K,N,gs", [(2176, 23552, 128), (4096, 28672, 128), (8576, 5888 + 256, -1), (896, 69632, 128)])
def test_gated(pkg, oracle, gpu, K, N, gs):
    pk, w = _case(pkg, oracle, gpu, K, N, gs, K + N)
    for M, dtype, act in [(5, "f16", "silu"), (16, "f16", "gelu"), (9, "bf16", "gelu_tanh"), (16, "bf16", "silu")]:
        assert pkg.ops.kernel_of(pk, M, DT[dtype], True) == "batch"
        x, bias = _rand(gpu, dtype, M, M, K) / 8, _rand(gpu, dtype, N, N)
        got = pkg.ops.linear_gate_up(pk, x, act, bias)
        assert all(torch.equal(got, pkg.ops.linear_gate_up(pk, x, act, bias)) for _ in range(3))
        sums = (x.double() @ w).to(DT[dtype]) + bias
        gate, up = sums.double().chunk(2, dim=1)
        f = {"silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu, "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}[act]
        want = f(gate).to(DT[dtype]).double() * up
        err = float((got.double() - want).abs().max() / want.abs().max())
        assert err <= {"f16": 2e-3, "bf16": 1.2e-2}[dtype]


def test_the_decode_path_runs_it_on_the_largest_layers(pkg, gpu):
    """Five and six rows of 2^28 weights and more stay the decode path's calls; their sums are those of seven rows' batch."""
    K, N, g = 8192, 32768, torch.Generator(device=gpu).manual_seed(1)
    words = lambda *s: torch.randint(-(2**31), 2**31 - 1, s, dtype=torch.int32, device=gpu, generator=g)  # noqa: E731
    pk = pkg.ops.make_packed(words(K, N // 8), words(K // 128, N // 8), (torch.rand((K // 128, N), device=gpu, generator=g) * 0.02).half(), None, 128, 1)
    x = _rand(gpu, "f16", 1, 7, K)
    seven = pkg.ops.linear(pk, x)
    for M in (5, 6):
        assert pkg.ops.kernel_of(pk, M) == "gemv"
        got = pkg.ops.linear(pk, x[:M])
        # (other K deals: fp32 sums in another order, so neighbouring outputs)
        assert float((got.double() - seven[:M].double()).abs().max() / seven.double().abs().max()) <= 2.0**-10


def test_without_a_workspace_the_batch_kernel_answers(pkg, oracle, gpu):
    """The C entry, no workspace: gate and up tiles could not meet."""
    import ctypes

    pk, w = _case(pkg, oracle, gpu, 4096, 12800, 128, 4)
    x = _rand(gpu, "f16", 1, 6, 4096)
    want = x.double() @ w
    out = torch.empty((6, 12800), device=gpu, dtype=torch.float16)
    lib = pkg._lib.load()
    rc = lib.q4_linear(ctypes.byref(pk.struct()), x.data_ptr(), None, out.data_ptr(), 6, 0, None, 0, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and float((out.double() - want).abs().max() / want.abs().max()) <= 2e-3


def test_replays(pkg, oracle, gpu):
    """Several replays of a graph with eager calls between them."""
    pk, w = _case(pkg, oracle, gpu, 4096, 28672, 128, 9)
    x = _rand(gpu, "f16", 1, 13, 4096) / 8
    want, want2 = pkg.ops.linear_gate_up(pk, x, "silu"), pkg.ops.linear(pk, x)
    pkg.ops.reserve_workspace(gpu, 16 << 20, pkg.ops.SHARED)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, out2 = pkg.ops.linear_gate_up(pk, x, "silu"), pkg.ops.linear(pk, x)
    for _ in range(4):
        out.zero_()
        out2.zero_()
        graph.replay()
        assert torch.equal(out, want) and torch.equal(out2, want2)
        assert torch.equal(pkg.ops.linear_gate_up(pk, x, "silu"), want)
        torch.cuda.synchronize()
