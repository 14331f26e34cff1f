"""Act-order batch decode kernel (q4_gemv_batch_act.cuh) at the edges of its row blocks, K deals and exchange levels, against
the oracle and against the kernels that a forced path runs.

Bars: max|y - ref| / max|ref| <= 2e-3 in fp16 (output rounding 2^-11 plus the fp32 accumulation), 8e-3 in bf16; gated 1.2e-2 in
bf16 (three roundings of 2^-8).
"""

import ctypes

import numpy as np
import pytest
import torch

from tests.util import max_rel_err, to_dev, to_f32

pytestmark = pytest.mark.gpu

TOL = {"f16": 2e-3, "bf16": 8e-3}
TOL_GATED = {"f16": 2e-3, "bf16": 1.2e-2}


def _weight(pkg, oracle, gpu, K, N, gs, seed, dtype, sym=False, g_idx=None):
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=seed, sym=sym, act_order=True)
    gi = gi if g_idx is None else g_idx
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), to_dev(gi, gpu), gs, 0)
    return pk, oracle.dequant_gptq(qw, qz, sc, gi, gs, dtype)


# K: one chunk per wave (4), ragged over the waves (9, 43), several exchange levels (32); tables of 4 to 128 groups
@pytest.mark.parametrize("K,N,gs,sym", [(512, 64, 128, False), (1152, 192, 32, False), (4096, 256, 128, True), (5504, 128, 128, False),
                                        (4096, 512, 32, False), (1024, 16384, 64, True)])
@pytest.mark.parametrize("M,dtype", [(1, "f16"), (6, "bf16"), (16, "f16"), (17, "bf16"), (32, "f16"), (33, "bf16"), (47, "f16"), (64, "bf16")])
def test_rows_and_shapes(pkg, oracle, gpu, K, N, gs, sym, M, dtype):
    pk, w = _weight(pkg, oracle, gpu, K, N, gs, K + N + M, dtype, sym)
    bf = dtype == "bf16"
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    b32 = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias = oracle.f32_to_bf16_bits(b32) if bf else b32.astype(np.float16)
    xt, bt = to_dev(x, gpu, bf16=bf), to_dev(bias, gpu, bf16=bf)
    y32, _ = oracle.linear_forward(x, w, bias, dtype)
    assert pkg.ops.kernel_of(pk, M, xt.dtype) == "batch"
    got = pkg.ops.linear(pk, xt, bt)
    assert torch.equal(got, pkg.ops.linear(pk, xt, bt))  # the exchange cells are left at zero
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]
    if N % 128 == 0:
        assert pkg.ops.kernel_of(pk, M, xt.dtype, True) == "batch"
        _, want = oracle.gate_up_forward(x, w, "silu", bias, dtype)
        gated = pkg.ops.linear_gate_up(pk, xt, "silu", bt)
        assert max_rel_err(to_f32(gated), oracle.to_f32(want, dtype)) <= TOL_GATED[dtype]
        assert torch.equal(gated, pkg.ops.linear_gate_up(pk, xt, "silu", bt, fused=True))
        two = pkg.ops.linear_gate_up(pk, xt, "silu", bt, fused=False)
        assert max_rel_err(to_f32(gated), to_f32(two)) <= TOL_GATED[dtype]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_one_hot_rows_read_the_weights_back(pkg, oracle, gpu, dtype):
    """Every weight is the reference's round_once(scale * (q - z)), with groups of any size and entries past the table clamped."""
    K, N, gs = 1024, 128, 64
    gi = np.random.default_rng(3).integers(0, K // gs, K).astype(np.int32)
    pk, w = _weight(pkg, oracle, gpu, K, N, gs, 5, dtype, g_idx=gi)
    bits = w.view(np.uint16)
    for at in range(0, K, 64):
        x = np.zeros((64, K), dtype=np.float32)
        x[np.arange(64), at + np.arange(64)] = 1.0
        xt = torch.from_numpy(x).to(gpu).to(torch.bfloat16 if dtype == "bf16" else torch.float16)
        got = pkg.ops.linear(pk, xt).cpu().view(torch.int16).numpy().view(np.uint16)
        want = bits[at:at + 64]
        assert np.array_equal(np.where(got == 0x8000, 0, got), np.where(want == 0x8000, 0, want))  # (a sum with -0 gives +0)


def test_infinite_activations_stay_in_their_row(pkg, oracle, gpu):
    pk, w = _weight(pkg, oracle, gpu, 4096, 256, 128, 7, "f16")
    x = to_dev(oracle.make_x(20, 4096, seed=8), gpu)
    clean = pkg.ops.linear(pk, x)
    x[7, 2048], x[19, 5] = float("inf"), float("nan")
    got = pkg.ops.linear(pk, x)
    ref = x[7, 2048].float().cpu() * torch.from_numpy(np.sign(w[2048].astype(np.float32)))
    assert torch.equal(torch.isnan(got[7].cpu()), torch.isnan(ref)) and torch.equal(torch.isposinf(got[7].cpu()), torch.isposinf(ref))
    assert torch.isnan(got[19]).all()
    keep = [r for r in range(20) if r not in (7, 19)]
    assert torch.equal(got[keep], clean[keep])


def test_without_a_workspace(pkg, oracle, gpu):
    """A call that the kernel would have to split for its LDS, without the cells of a split: another kernel's, as before."""
    import ctypes

    K, N, M = 27264, 128, 64  # 426 groups: their table and the groups of all rows are more than a workgroup's LDS
    pk, w = _weight(pkg, oracle, gpu, K, N, 64, 11, "f16")
    assert pkg.ops.kernel_of(pk, M) == "batch"  # (with the cells it is this kernel's)
    x = oracle.make_x(M, K, seed=12)
    xt, y = to_dev(x, gpu), torch.empty((M, N), dtype=torch.float16, device=gpu)
    lib = pkg._lib
    lib.check(lib.load().q4_linear(ctypes.byref(pk.struct()), xt.data_ptr(), None, y.data_ptr(), M, 0, None, 0,
                                   torch.cuda.current_stream().cuda_stream))
    y32, _ = oracle.linear_forward(x, w, None, "f16")
    assert max_rel_err(to_f32(y), y32) <= TOL["f16"]


def test_replays(pkg, oracle, gpu):
    """A captured call, replayed with the program's own calls in between."""
    pk, _ = _weight(pkg, oracle, gpu, 4096, 512, 128, 9, "f16")
    pk.prepare()
    x = to_dev(oracle.make_x(24, 4096, seed=8), gpu)
    want = pkg.ops.linear(pk, x), pkg.ops.linear_gate_up(pk, x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = pkg.ops.linear(pk, x), pkg.ops.linear_gate_up(pk, x)
    for _ in range(4):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, want))
        assert torch.equal(pkg.ops.linear(pk, x), want[0])


@pytest.mark.parametrize("K,N,gs", [(4096, 28672, 128), (2048, 24576, 64), (2176, 49152, 128), (5504, 192, 128), (4608, 4608, 128), (18944, 256, 256), (8192, 1280, 32), (2304, 1152, 32)])
@pytest.mark.parametrize("M,dtype", [(1, "f16"), (3, "bf16"), (4, "f16"), (5, "f16"), (16, "f16"), (37, "bf16")])
@pytest.mark.parametrize("sym", [False, True])
def test_tiles_and_splits(pkg, oracle, gpu, K, N, gs, M, dtype, sym):
    """128-column tiles of the gated epilogue in one round and in workgroups along K, x of a few rows through LDS over long ranges, splits
    that are no power of two; one zero point and several."""
    if K * N * M > 2.5e9:
        M = 5 if M == 37 else M
    bf = dtype == "bf16"
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=K + M, sym=sym, act_order=True)
    w = oracle.dequant_gptq(qw, qz, sc, gi, gs, dtype)
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), to_dev(gi, gpu), gs, 0)
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    xt = to_dev(x, gpu, bf16=bf)
    y32, _ = oracle.linear_forward(x, w, None, dtype)
    got = pkg.ops.linear(pk, xt)
    assert torch.equal(got, pkg.ops.linear(pk, xt))
    assert max_rel_err(to_f32(got), y32) <= (8e-3 if bf else 2e-3)
    if N % 128 == 0:
        _, want = oracle.gate_up_forward(x, w, "silu", None, dtype)
        gated = pkg.ops.linear_gate_up(pk, xt, "silu")
        assert torch.equal(gated, pkg.ops.linear_gate_up(pk, xt, "silu"))
        assert max_rel_err(to_f32(gated), oracle.to_f32(want, dtype)) <= (1.2e-2 if bf else 2e-3)
    # one-hot rows read the rounded weights back bit for bit
    hot = torch.zeros_like(xt)
    ks = (torch.arange(M) * 997 + 13) % K
    hot[torch.arange(M), ks] = 1
    back = pkg.ops.linear(pk, hot).cpu().view(torch.int16).numpy().view(np.uint16)
    assert np.array_equal(back & 0x7FFF, w[ks.numpy()].view(np.uint16) & 0x7FFF)  # (a zero may have lost its sign)


@pytest.mark.parametrize("M", [1, 4, 16])
@pytest.mark.parametrize("sym", [False, True])
def test_wide_gated_tiles_in_workgroups_along_k(pkg, gpu, M, sym):
    """128-column tiles beyond one a CU: against the plain launch on 64 columns and the elementwise kernel, whose roundings are the same and whose
    fp32 sums are in another order, so that an output is off by its sums' last place (2^-11 each) now and then."""
    K, N, gs, g = 5120, 49152, 128, torch.Generator(device=gpu).manual_seed(M)
    words = lambda *s: torch.randint(-(2**31), 2**31 - 1, s, dtype=torch.int32, device=gpu, generator=g)  # noqa: E731
    qz = torch.full((K // gs, N // 8), 0x77777777, dtype=torch.int32, device=gpu) if sym else words(K // gs, N // 8)
    sc = (torch.rand((K // gs, N), device=gpu, generator=g) * 0.01 + 0.001).half()
    g_idx = (torch.arange(K, device=gpu) // gs)[torch.randperm(K, device=gpu, generator=g)].to(torch.int32)
    pk = pkg.ops.make_packed(words(K // 8, N), qz, sc, g_idx, gs, 0)
    tiles = (ctypes.c_int * 4)()
    assert pkg._lib.load().q4_linear_tiles(ctypes.byref(pk.struct()), M, 0, 1, tiles) == 0 and tiles[1] == 128 and tiles[3] > 1
    x = (torch.randn((M, K), device=gpu, generator=g) / 16).half()
    got, sums = pkg.ops.linear_gate_up(pk, x, "silu"), pkg.ops.linear(pk, x)
    assert torch.equal(got, pkg.ops.linear_gate_up(pk, x, "silu"))
    want, (gate, up) = pkg.ops.act_mul(sums, "silu").double(), sums.double().chunk(2, dim=1)
    # the sums' last place through the product (slope of silu at most 1.1), and the two roundings behind them
    bar = 2.0**-10 * (1.1 * gate.abs() * up.abs() + torch.nn.functional.silu(gate).abs() * up.abs()) + 2.0**-9 * want.abs() + 2.0**-24
    assert bool(((got.double() - want).abs() <= bar).all())
    assert float((got != want).double().mean()) < 0.05
