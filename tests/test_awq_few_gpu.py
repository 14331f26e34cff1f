"""AWQ decode kernel for one to four rows (q4_gemv_awq_few.cuh) at the edges of its tiles, K deals and exchange levels.

Bars: the sums are those of x (q - z), scaled, in fp32; an output is off by its own rounding (2^-11 of it in fp16, 2^-8 in bf16) and by
fp32 sums, of which a chunk's 32 MFMA of four K rows and K / 128 chunks follow each other: 36 + K / 128 roundings of 2^-24 of the
sum of the terms' magnitudes.  Gated: three roundings follow each other (sums, activation, product).
"""

import numpy as np
import pytest
import torch

from tests.util import max_rel_err, to_dev, to_f32

pytestmark = pytest.mark.gpu

DT = {"f16": torch.float16, "bf16": torch.bfloat16}
U = {"f16": 2.0**-11, "bf16": 2.0**-8}


def _case(pkg, oracle, gpu, K, N, gs, seed):
    g = K if gs == -1 else gs
    qw, qz, sc = oracle.make_awq(K, N, g, seed=seed)
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 1)
    ints = oracle.dequant_awq(qw, qz, np.ones_like(sc), g, "f16").astype(np.float64)
    w = torch.from_numpy(ints * np.repeat(sc.astype(np.float64), g, axis=0)).to(gpu)
    return pk, w


# K: one chunk a wave, ragged deals (17, 43, 67 chunks), an odd number of workgroups along K; N: one tile, an odd number, pairs of tiles
@pytest.mark.parametrize("K,N,gs", [(2048, 256, 128), (2176, 768, 128), (5504, 512, 256), (8576, 1280, 128), (4096, 28672, 128), (14336, 4096, -1),
                                    (8192, 10240, 512), (2176, 16640, 128), (5504, 6400, 128), (4992, 4096, 128)])
@pytest.mark.parametrize("M,dtype", [(1, "f16"), (1, "bf16"), (2, "f16"), (3, "bf16"), (4, "f16"), (4, "bf16")])
def test_plain(pkg, oracle, gpu, K, N, gs, M, dtype):
    gs = gs if gs == -1 or K % gs == 0 else 128
    pk, w = _case(pkg, oracle, gpu, K, N, gs, K + M)
    x = torch.randn((M, K), device=gpu, generator=torch.Generator(device=gpu).manual_seed(M)).to(DT[dtype])
    bias = torch.randn(N, device=gpu, generator=torch.Generator(device=gpu).manual_seed(N)).to(DT[dtype])
    got = pkg.ops.linear(pk, x)
    assert all(torch.equal(got, pkg.ops.linear(pk, x)) for _ in range(3))  # cells left at zero, no order of arrival in the sums
    want, terms = x.double() @ w, x.double().abs() @ w.abs()
    assert bool(((got.double() - want).abs() <= U[dtype] * want.abs() + (36 + K // 128) * 2.0**-24 * terms + 2.0**-25).all())
    assert torch.equal(pkg.ops.linear(pk, x, bias), got + bias)
    # an infinity, a NaN and a large value under other rows
    x[0, K // 2] = float("inf")
    if M > 1:
        x[M - 1, 5] = float("nan")
    bad = pkg.ops.linear(pk, x).float()
    wcol = w[K // 2]
    assert bool((torch.where(wcol == 0, torch.isnan(bad[0]), bad[0] == torch.sign(wcol).float() * float("inf"))).all())
    assert M == 1 or bool(torch.isnan(bad[M - 1]).all())
    assert torch.equal(bad[1 : max(1, M - 1)], got.float()[1 : max(1, M - 1)])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_large_activation_under_zero_weights(pkg, oracle, gpu, dtype):
    """Nothing of it reaches the sums: the zero point leaves the weights before they meet x."""
    K, N = 4096, 512
    qw, qz, sc = oracle.make_awq(K, N, 128, seed=3)
    q, z = oracle.awq_unpack_cols(qw), oracle.awq_unpack_cols(qz)
    q[300] = z[300 // 128]
    pk = pkg.ops.make_packed(to_dev(oracle.awq_pack_cols(q), gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, 128, 1)
    x = torch.randn((2, K), device=gpu, generator=torch.Generator(device=gpu).manual_seed(1)).to(DT[dtype])
    x[1, 300] = 0
    clean = pkg.ops.linear(pk, x)
    x[1, 300] = 6e4 if dtype == "f16" else 2.0**100
    assert torch.equal(pkg.ops.linear(pk, x), clean)


@pytest.mark.parametrize("K,N,gs", [(2176, 512, 128), (4096, 28672, 128), (4096, 22016, 256), (8576, 1536, 128), (3584, 37888, 128)])
@pytest.mark.parametrize("M,dtype,act", [(1, "f16", "silu"), (2, "f16", "gelu"), (4, "f16", "gelu_tanh"), (1, "bf16", "silu"), (3, "bf16", "silu")])
def test_gated(pkg, oracle, gpu, K, N, gs, M, dtype, act):
    g = gs if K % gs == 0 else 128
    qw, qz, sc = oracle.make_awq(K, N, g, seed=K + N)
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 1)
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    b32 = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias = oracle.f32_to_bf16_bits(b32) if dtype == "bf16" else b32.astype(np.float16)
    _, want = oracle.gate_up_forward(x, oracle.dequant_awq(qw, qz, sc, g, dtype), act, bias, dtype)
    xt, bt = to_dev(x, gpu, bf16=dtype == "bf16"), to_dev(bias, gpu, bf16=dtype == "bf16")
    got = pkg.ops.linear_gate_up(pk, xt, act, bt)
    assert torch.equal(got, pkg.ops.linear_gate_up(pk, xt, act, bt))
    # (against weights rounded one by one: 3 x 2^-8 and 3 x 2^-11, the latter inside the 2e-3 of the other parity tests)
    assert max_rel_err(to_f32(got), oracle.to_f32(want, dtype)) <= {"f16": 2e-3, "bf16": 1.2e-2}[dtype]


# ragged deals of K (17 and 67 chunks) over as many tiles as this kernel takes them for
@pytest.mark.parametrize("K,N", [(2176, 20480), (8576, 5120)])
@pytest.mark.parametrize("M,dtype", [(1, "f16"), (3, "bf16"), (4, "f16")])
def test_gated_against_64_bits(pkg, oracle, gpu, K, N, M, dtype):
    """Bar: the roundings of both sums, of the activation (whose slope is at most 1.1) and of the product, one unit each, and the fp32 sums'
    36 + K / 128; 1 % for their products."""
    pk, w = _case(pkg, oracle, gpu, K, N, 128, K + N)
    x = (torch.randn((M, K), device=gpu, generator=torch.Generator(device=gpu).manual_seed(M)) / 8).to(DT[dtype])
    got, u = pkg.ops.linear_gate_up(pk, x, "silu"), U[dtype]
    sums, terms = x.double() @ w, (x.double().abs() @ w.abs()) * (36 + K // 128) * 2.0**-24
    gate, up = sums.chunk(2, dim=1)
    eg, eu = (u * sums.abs() + terms).chunk(2, dim=1)
    act = torch.nn.functional.silu(gate)
    bar = 1.1 * eg * up.abs() + act.abs() * eu + 2 * u * (act * up).abs()
    assert bool(((got.double() - act * up).abs() <= 1.01 * bar + 2.0**-24).all())


def test_replays_and_captures(pkg, oracle, gpu):
    """Several replays of a graph with eager calls between them, and a stream of their own."""
    pk, w = _case(pkg, oracle, gpu, 4096, 4096, 128, 9)
    x = torch.randn((3, 4096), device=gpu).half()
    want = pkg.ops.linear(pk, x)
    pkg.ops.reserve_workspace(gpu, 16 << 20, pkg.ops.SHARED)
    graph, out = torch.cuda.CUDAGraph(), None
    with torch.cuda.graph(graph):
        out = pkg.ops.linear(pk, x)
    for _ in range(4):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want)
        assert torch.equal(pkg.ops.linear(pk, x), want)
        torch.cuda.synchronize()
