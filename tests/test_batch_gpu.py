"""Batch decode kernel (q4_gemv_batch.cuh) at the edges of its row blocks, wave tiles, K deals and
exchange levels, against the oracle.

Bars as in the other parity tests: max|y - ref| / max|ref| <= 2e-3 in fp16 (output rounding 2^-11 plus
the fp32 accumulation), 8e-3 in bf16 (output rounding 2^-8).  The gated epilogue rounds three times (gate and
up sums, activation, product), and where the kernel leaves the weights unrounded each of them can fall on the
neighbouring value: 3 x 2^-8 = 1.2e-2 in bf16, 3 x 2^-11 = 1.5e-3 in fp16 (inside its bar).
"""

import numpy as np
import pytest
import torch

from tests.util import max_rel_err, to_dev, to_f32

pytestmark = pytest.mark.gpu

TOL = {"f16": 2e-3, "bf16": 8e-3}
TOL_GATED = {"f16": 2e-3, "bf16": 1.2e-2}


def _weight(pkg, oracle, gpu, layout, K, N, gs, seed, dtype):
    g = K if gs == -1 else gs
    if layout == "awq":
        qw, qz, sc = oracle.make_awq(K, N, g, seed=seed)
        return pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 1), oracle.dequant_awq(qw, qz, sc, g, dtype)
    qw, qz, sc, _ = oracle.make_gptq(K, N, g, seed=seed, sym=False)
    return pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, g, 0), oracle.dequant_gptq(qw, qz, sc, None, g, dtype)


# K in chunks of 128 rows: fewest (4), ragged over the waves (9, 43), two and more exchange levels (32);
# N: one wave tile, several, tiles that pair up on one XCD (AWQ: 2048 = 16 tiles), no splits (16384)
SHAPES = [("gptq", 512, 64, 128), ("gptq", 1152, 192, 64), ("gptq", 4096, 256, 128), ("gptq", 5504, 512, 128),
          ("gptq", 1024, 16384, 256), ("gptq", 1024, 128, -1), ("awq", 512, 256, 64), ("awq", 1152, 512, 128),
          ("awq", 4096, 2048, 128), ("awq", 5504, 256, 128)]


@pytest.mark.parametrize("layout,K,N,gs", SHAPES)
@pytest.mark.parametrize("M,dtype", [(1, "bf16"), (5, "f16"), (16, "bf16"), (17, "f16"), (32, "f16"), (33, "bf16"), (48, "f16"), (49, "f16"), (64, "bf16")])
def test_rows_and_shapes(pkg, oracle, gpu, layout, K, N, gs, M, dtype):
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, gs, K // 128 + N + M, dtype)
    bf = dtype == "bf16"
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    b32 = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias = oracle.f32_to_bf16_bits(b32) if bf else b32.astype(np.float16)
    y32, _ = oracle.linear_forward(x, w, bias, dtype)
    # (AWQ beyond 48 rows belongs to the prefill kernels)
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16 if bf else torch.float16) == ("gemm" if layout == "awq" and M > 48 else "batch")
    xt, bt = to_dev(x, gpu, bf16=bf), to_dev(bias, gpu, bf16=bf)
    got = pkg.ops.linear(pk, xt, bt)
    again = pkg.ops.linear(pk, xt, bt)  # the exchange cells are left at zero, the order of arrival does not matter
    torch.cuda.synchronize()
    assert torch.equal(got, again)
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]


@pytest.mark.parametrize("layout,K,N", [("gptq", 512, 128), ("gptq", 1152, 384), ("gptq", 4096, 512), ("gptq", 1024, 32768),
                                        ("awq", 512, 256), ("awq", 4096, 1024), ("awq", 1152, 8192)])
@pytest.mark.parametrize("M,dtype", [(1, "f16"), (7, "bf16"), (16, "f16"), (23, "bf16"), (32, "f16"), (47, "bf16"), (63, "f16")])
def test_gated_epilogue(pkg, oracle, gpu, layout, K, N, M, dtype):
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, 128, K + N + M, dtype)
    bf = dtype == "bf16"
    x = oracle.make_x(M, K, seed=M + 1, dtype=dtype)
    b32 = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias = oracle.f32_to_bf16_bits(b32) if bf else b32.astype(np.float16)
    _, want = oracle.gate_up_forward(x, w, "silu", bias, dtype)
    got = pkg.ops.linear_gate_up(pk, to_dev(x, gpu, bf16=bf), "silu", to_dev(bias, gpu, bf16=bf))
    assert max_rel_err(to_f32(got), oracle.to_f32(want, dtype)) <= TOL_GATED[dtype]


@pytest.mark.parametrize("layout,K,N", [("gptq", 4096, 256), ("awq", 4096, 512)])
def test_non_finite_rows_stay_alone(pkg, oracle, gpu, layout, K, N):
    """An infinite activation makes its own row what fp32 arithmetic makes it, through every exchange
    level, and leaves the other rows alone; a row of zeros gives +0."""
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, 128, 3, "f16")
    x = oracle.make_x(20, K, seed=8)
    x[4] = 0
    clean = pkg.ops.linear(pk, to_dev(x, gpu)).cpu().numpy()
    assert not clean[4].view(np.uint16).any()
    x[7, K // 2] = np.inf
    x[19, 5] = np.nan
    got = pkg.ops.linear(pk, to_dev(x, gpu)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        ref = x[[7]].astype(np.float32) @ w.astype(np.float32)
    assert np.array_equal(np.isnan(got[7]), np.isnan(ref[0])) and np.array_equal(np.isposinf(got[7]), np.isposinf(ref[0]))
    assert np.isnan(got[19]).all()
    keep = [r for r in range(20) if r not in (7, 19)]
    assert np.array_equal(got[keep], clean[keep])


@pytest.mark.parametrize("M,dtype", [(1, "f16"), (2, "bf16"), (4, "f16")])
def test_few_rows_with_groups_of_64(pkg, oracle, gpu, M, dtype):
    """One to four rows run here for groups of 64 rows (the last group ragged over the K waves)."""
    pk, w = _weight(pkg, oracle, gpu, "gptq", 1152, 4096, 64, M, dtype)
    x = oracle.make_x(M, 1152, seed=M, dtype=dtype)
    y32, _ = oracle.linear_forward(x, w, None, dtype)
    got = pkg.ops.linear(pk, to_dev(x, gpu, bf16=dtype == "bf16"))
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]


# (layers beyond 2^25 weights, on each side of the rule: the output's rounding 2^-11, 2^-8 and its share in the gated product)
@pytest.mark.parametrize("K,N,gs,M,dtype,gated,kernel", [
    (11008, 4096, 128, 1, "bf16", False, "batch"), (11008, 4096, 128, 4, "f16", False, "batch"), (11008, 4096, 128, 3, "f16", False, "gemv"),
    (8320, 4352, 64, 3, "f16", False, "batch"), (8320, 4352, 32, 1, "f16", False, "batch"), (4096, 12288, 128, 2, "bf16", False, "gemv"),
    (2176, 15488, 128, 1, "f16", False, "batch"), (8320, 4224, 32, 2, "bf16", False, "batch"),
    (8448, 384, 128, 33, "f16", False, "batch"), (8448, 512, 128, 33, "f16", False, "gemm"), (1152, 7168, 128, 1, "f16", True, "batch"), (2048, 17408, 128, 3, "bf16", True, "batch")])
def test_few_awq_rows(pkg, oracle, gpu, K, N, gs, M, dtype, gated, kernel):
    pk, w = _weight(pkg, oracle, gpu, "awq", K, N, gs, M, dtype)
    bf = dtype == "bf16"
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16 if bf else torch.float16, gated) == kernel
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    xt = to_dev(x, gpu, bf16=bf)
    if gated:
        _, want = oracle.gate_up_forward(x, w, "silu", None, dtype)
        got = pkg.ops.linear_gate_up(pk, xt, "silu")
        assert max_rel_err(to_f32(got), oracle.to_f32(want, dtype)) <= TOL_GATED[dtype]
    else:
        y32, _ = oracle.linear_forward(x, w, None, dtype)
        got = pkg.ops.linear(pk, xt)
        assert max_rel_err(to_f32(got), y32) <= TOL[dtype]


@pytest.mark.parametrize("layout,N,M,dtype", [("gptq", 512, 13, "bf16"), ("gptq", 512, 37, "f16"), ("gptq", 512, 64, "bf16"),
                                              ("gptq", 32768, 16, "f16"), ("awq", 512, 6, "bf16"), ("awq", 512, 32, "f16")])
def test_weights_are_not_rounded(pkg, oracle, gpu, layout, N, M, dtype):
    """Against 64-bit sums of scale * (q - z) only the output's rounding is left: its relative 2-norm is
    0.41 to 0.43 u (u = 2^-11, 2^-8; values spread over their binade), with rounded weights 0.59 u; the bar
    is half way."""
    _unrounded(pkg, oracle, gpu, layout, 2048, N, M, dtype)


@pytest.mark.parametrize("K,N,M", [(768, 17408, 33), (512, 16640, 48), (896, 17408, 40)])
def test_weights_of_small_wide_matrices_are_not_rounded(pkg, oracle, gpu, K, N, M):
    """Three row blocks on matrices small enough for the decode kernels, which carry the scale to the sums."""
    assert pkg.ops.select_path(pkg.ops.make_packed(*[to_dev(a, gpu) for a in oracle.make_gptq(K, N, 128, seed=1)[:3]], None, 128, 0), M) == "gemv"
    _unrounded(pkg, oracle, gpu, "gptq", K, N, M, "f16")


def _unrounded(pkg, oracle, gpu, layout, K, N, M, dtype):
    gs = 128
    if layout == "awq":
        qw, qz, sc = oracle.make_awq(K, N, gs, seed=N + M)
        deq = oracle.dequant_awq
    else:
        qw, qz, sc, _ = oracle.make_gptq(K, N, gs, seed=N + M, sym=False)
        deq = lambda a, b, c, g, d: oracle.dequant_gptq(a, b, c, None, g, d)  # noqa: E731
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, gs, 1 if layout == "awq" else 0)
    ints = np.asarray(deq(qw, qz, np.ones_like(sc), gs, "f16")).astype(np.float64)
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    xt = to_dev(x, gpu, bf16=dtype == "bf16")
    want = xt.double().cpu().numpy() @ (ints * np.repeat(sc.astype(np.float64), gs, axis=0))
    err = np.linalg.norm(pkg.ops.linear(pk, xt).double().cpu().numpy() - want) / np.linalg.norm(want)
    assert err <= 0.51 * (2.0**-8 if dtype == "bf16" else 2.0**-11)


@pytest.mark.parametrize("T,E,dtype", [(52, 4, "f16"), (64, 4, "bf16"), (30, 2, "f16"), (48, 2, "bf16")])
def test_weights_of_few_experts_are_not_rounded(pkg, oracle, gpu, T, E, dtype):
    """Grouped launches of up to 64 tokens with three and four row blocks an expert, on wide matrices."""
    K, N, gs, topk = 1024, 16384, 128, 2
    parts = [oracle.make_gptq(K, N, gs, seed=E + e, sym=False)[:3] for e in range(E)]
    packed = pkg.ops.make_packed_moe(*[torch.stack([to_dev(p[i], gpu) for p in parts]) for i in range(3)], gs)
    x = to_dev(oracle.make_x(T, K, seed=T, dtype=dtype), gpu, bf16=dtype == "bf16")
    routing = pkg.ops.moe_route(torch.randn((T, E), device=gpu, generator=torch.Generator(device=gpu).manual_seed(T)), topk)
    got = pkg.ops.moe_linear(packed, x, routing, gather=True).double().cpu().numpy()
    rows, offsets = routing.sorted_tokens.cpu().numpy(), routing.expert_offsets.cpu().numpy()
    want = np.empty_like(got)
    for e, (qw, qz, sc) in enumerate(parts):
        w = np.asarray(oracle.dequant_gptq(qw, qz, np.ones_like(sc), None, gs, "f16")).astype(np.float64) * np.repeat(sc.astype(np.float64), gs, axis=0)
        own = slice(offsets[e], offsets[e + 1])
        want[own] = x.double().cpu().numpy()[rows[own]] @ w
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 0.51 * (2.0**-8 if dtype == "bf16" else 2.0**-11)


@pytest.mark.parametrize("layout,K,N,M", [("gptq", 2048, 512, 1), ("gptq", 2048, 512, 16), ("gptq", 4096, 256, 37), ("gptq", 1152, 192, 64),
                                          ("gptq", 1024, 32768, 20), ("awq", 2048, 512, 4), ("awq", 4096, 512, 24)])
@pytest.mark.parametrize("kind", ["dc_offset", "one_sign", "outliers", "small", "silu_product"])
def test_bf16_off_distribution(pkg, oracle, gpu, layout, K, N, M, kind):
    """bf16 sums of the exact integers q - z on activations whose sum is far from zero.  Against 64-bit sums with unrounded weights
    an output is off by its own rounding (8 significant bits: 2^-8 of it), and by fp32 sums of the terms x (q - z) scale, of which a
    stage's 64 pass two MFMA of 32 and K / 64 stages follow: 2 + 32 + K / 64 roundings of 2^-24 of the terms' sum."""
    from tests.test_offdist_gpu import make_activations

    gs = 128 if K % 256 == 0 else 64
    if layout == "awq":
        qw, qz, sc = oracle.make_awq(K, N, gs, seed=M)
        ints = oracle.dequant_awq(qw, qz, np.ones_like(sc), gs, "f16")
    else:
        qw, qz, sc, _ = oracle.make_gptq(K, N, gs, seed=M, sym=False)
        ints = oracle.dequant_gptq(qw, qz, np.ones_like(sc), None, gs, "f16")
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, gs, 1 if layout == "awq" else 0)
    x = torch.from_numpy(make_activations(kind, M, K, M)).to(gpu).bfloat16()
    got = pkg.ops.linear(pk, x).double()
    scale = torch.from_numpy(np.repeat(sc.astype(np.float64), gs, axis=0)).to(gpu)
    w = torch.from_numpy(np.asarray(ints).astype(np.float64)).to(gpu) * scale
    want, terms = x.double() @ w, x.double().abs() @ w.abs()
    assert bool(((got - want).abs() <= 2.0**-8 * want.abs() + (34 + K // 64) * 2.0**-24 * terms).all())


@pytest.mark.parametrize("layout", ["gptq", "awq"])
@pytest.mark.parametrize("gs,M", [(128, 3), (128, 32), (64, 13), (32, 13)])
@pytest.mark.parametrize("value", [2.0**30, 2.39e36])
def test_bf16_sums_meet_x_times_weight_alone(pkg, oracle, gpu, layout, gs, M, value):
    """A large activation under weights that are zero, but for one column: nothing of it may reach the other sums, and its product,
    finite in fp32, stays finite.  Bound as above; the large row's term is zero where its weight is."""
    K, N = 1024, 512
    if layout == "awq":
        qw, qz, sc = oracle.make_awq(K, N, gs, seed=M)
        q, z = oracle.awq_unpack_cols(qw), oracle.awq_unpack_cols(qz)
        z[300 // gs] = 8
        q[300], q[300, 77] = 8, 15
        qw, qz = oracle.awq_pack_cols(q), oracle.awq_pack_cols(z)
        ints = oracle.dequant_awq(qw, qz, np.ones_like(sc), gs, "f16")
    else:
        qw, qz, sc, _ = oracle.make_gptq(K, N, gs, seed=M, sym=True)
        q = oracle.unpack_rows(qw)
        q[300], q[300, 77] = 8, 15
        qw = oracle.pack_rows(q)
        ints = oracle.dequant_gptq(qw, qz, np.ones_like(sc), None, gs, "f16")
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, gs, 1 if layout == "awq" else 0)
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16) == "batch"
    x = to_dev(oracle.make_x(M, K, seed=M, dtype="bf16"), gpu, bf16=True)
    x[1, 300] = value
    got = pkg.ops.linear(pk, x).double()
    w = torch.from_numpy(np.asarray(ints).astype(np.float64) * np.repeat(sc.astype(np.float64), gs, axis=0)).to(gpu)
    assert int((w[300] != 0).sum()) == 1
    want, terms = x.double() @ w, x.double().abs() @ w.abs()
    assert bool(torch.isfinite(got).all())
    assert bool(((got - want).abs() <= 2.0**-8 * want.abs() + (34 + K // 32) * 2.0**-24 * terms).all())


@pytest.mark.parametrize("layout,K,N,gs", [("gptq", 4096, 256, 128), ("gptq", 1152, 192, 64), ("gptq", 1024, 32768, 128), ("awq", 4096, 512, 128)])
@pytest.mark.parametrize("M", [3, 20, 37, 61])
def test_bf16_non_finite_rows_stay_alone(pkg, oracle, gpu, layout, K, N, gs, M):
    """Infinite and NaN activations keep the class that fp32 arithmetic on the weights gives them, the other rows keep their bits."""
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, gs, 3, "bf16")
    x = to_dev(oracle.make_x(M, K, seed=8, dtype="bf16"), gpu, bf16=True)
    clean = pkg.ops.linear(pk, x)
    x[1, K // 2], x[M - 1, 5] = float("inf"), float("nan")
    if M > 3:
        x[M - 2, 7], x[M - 2, K - 1] = float("-inf"), float("inf")
    got = pkg.ops.linear(pk, x).float().cpu().numpy()
    poisoned = [1, M - 1] + ([M - 2] if M > 3 else [])
    with np.errstate(invalid="ignore"):
        for r in poisoned:
            ref = (x[r].float().cpu().numpy()[:, None] * oracle.to_f32(w, "bf16")).sum(axis=0)
            assert np.array_equal(np.isnan(got[r]), np.isnan(ref)) and np.array_equal(np.isposinf(got[r]), np.isposinf(ref))
            assert not np.isfinite(got[r]).any()
    keep = [r for r in range(M) if r not in poisoned]
    assert np.array_equal(got[keep], clean.float().cpu().numpy()[keep])


@pytest.mark.parametrize("K,N,M", [(8192, 8192, 1), (16384, 4096, 3), (8192, 8192, 2)])
def test_bf16_few_rows_on_large_layers(pkg, oracle, gpu, K, N, M):
    """One to three bf16 rows on 2^26 weights and more, plain and gated: the decode kernels'."""
    pk, w = _weight(pkg, oracle, gpu, "gptq", K, N, 128, M, "bf16")
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16) == "gemv" and pkg.ops.kernel_of(pk, M, torch.bfloat16, True) == ("none" if M == 3 else "gemv")
    x = oracle.make_x(M, K, seed=M, dtype="bf16")
    y32, _ = oracle.linear_forward(x, w, None, "bf16")
    assert max_rel_err(to_f32(pkg.ops.linear(pk, to_dev(x, gpu, bf16=True))), y32) <= TOL["bf16"]
    _, want = oracle.gate_up_forward(x, w, "silu", None, "bf16")
    got = pkg.ops.linear_gate_up(pk, to_dev(x, gpu, bf16=True), "silu")
    assert max_rel_err(to_f32(got), oracle.to_f32(want, "bf16")) <= TOL_GATED["bf16"]


@pytest.mark.parametrize("layout,K,N", [("gptq", 512, 64), ("gptq", 1152, 384), ("gptq", 1024, 16384), ("gptq", 2048, 16384), ("awq", 512, 256), ("awq", 4096, 1024),
                                        ("awq", 9216, 512)])
@pytest.mark.parametrize("M,dtype", [(1, "f16"), (3, "bf16"), (16, "f16"), (17, "bf16"), (32, "f16"), (33, "bf16"), (48, "f16"), (64, "bf16")])
def test_groups_of_32_rows(pkg, oracle, gpu, layout, K, N, M, dtype):
    """A scale and a zero point per MFMA step: plain, gated, and rows that are not finite."""
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, 32, K + M, dtype)
    bf = dtype == "bf16"
    td = torch.bfloat16 if bf else torch.float16
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    xt = to_dev(x, gpu, bf16=bf)
    assert pkg.ops.kernel_of(pk, M, td) == ("batch" if layout == "gptq" or M <= 48 else "gemm")
    y32, _ = oracle.linear_forward(x, w, None, dtype)
    got = pkg.ops.linear(pk, xt)
    assert torch.equal(got, pkg.ops.linear(pk, xt))
    assert max_rel_err(to_f32(got), y32) <= TOL[dtype]
    if N % 128 == 0:
        _, want = oracle.gate_up_forward(x, w, "silu", None, dtype)
        gated = pkg.ops.linear_gate_up(pk, xt, "silu")
        assert max_rel_err(to_f32(gated), oracle.to_f32(want, dtype)) <= TOL_GATED[dtype]
    xt[M - 1, 5] = float("inf")
    bad = pkg.ops.linear(pk, xt)
    ref = xt[M - 1, 5].float().cpu() * torch.from_numpy(np.sign(oracle.to_f32(w, dtype)[5]))
    want = torch.where(ref == ref, ref, torch.full_like(ref, float("nan")))  # (an infinity times zero)
    assert torch.equal(torch.isnan(bad[M - 1].float().cpu()), torch.isnan(want))
    assert torch.equal(torch.isposinf(bad[M - 1].float().cpu()), torch.isposinf(want)) and torch.equal(bad[:-1], got[:-1])


@pytest.mark.parametrize("layout,N", [("gptq", 192), ("gptq", 16640), ("awq", 512)])
@pytest.mark.parametrize("K,gs", [(640, 64), (640, 128), (1408, 128), (1280, 256), (1152, -1)])
@pytest.mark.parametrize("M,dtype", [(6, "f16"), (16, "bf16"), (31, "f16"), (40, "bf16")])
def test_group_lengths_over_ragged_deals(pkg, oracle, gpu, layout, N, K, gs, M, dtype):
    """Groups that end inside, with and beyond a 128-row chunk, K waves that walk one chunk and several."""
    pk, w = _weight(pkg, oracle, gpu, layout, K, N, gs, K + M, dtype)
    bf = dtype == "bf16"
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    assert pkg.ops.kernel_of(pk, M, torch.bfloat16 if bf else torch.float16) == "batch"
    y32, _ = oracle.linear_forward(x, w, None, dtype)
    assert max_rel_err(to_f32(pkg.ops.linear(pk, to_dev(x, gpu, bf16=bf))), y32) <= TOL[dtype]


@pytest.mark.parametrize("T,dtype", [(9, "f16"), (40, "bf16")])
def test_experts_in_groups_of_64(pkg, oracle, gpu, T, dtype):
    K, N, E, gs, topk = 640, 768, 4, 64, 2
    parts = [oracle.make_gptq(K, N, gs, seed=e, sym=False)[:3] for e in range(E)]
    packed = pkg.ops.make_packed_moe(*[torch.stack([to_dev(p[i], gpu) for p in parts]) for i in range(3)], gs)
    xs = oracle.make_x(T, K, seed=T, dtype=dtype)
    routing = pkg.ops.moe_route(torch.randn((T, E), device=gpu, generator=torch.Generator(device=gpu).manual_seed(T)), topk)
    got = to_f32(pkg.ops.moe_linear(packed, to_dev(xs, gpu, bf16=dtype == "bf16"), routing, gather=True))
    rows, offsets = routing.sorted_tokens.cpu().numpy(), routing.expert_offsets.cpu().numpy()
    for e, (qw, qz, sc) in enumerate(parts):
        own = slice(offsets[e], offsets[e + 1])
        if own.start < own.stop:
            want, _ = oracle.linear_forward(xs[rows[own]], oracle.dequant_gptq(qw, qz, sc, None, gs, dtype), None, dtype)
            assert max_rel_err(got[own], want) <= TOL[dtype]


@pytest.mark.parametrize("K,N,M,dtype", [(16640, 192, 13, "bf16"), (16640, 192, 37, "f16"), (2176, 16384, 37, "f16"), (2176, 16384, 5, "f16"),
                                         (2176, 32768, 20, "bf16"), (3200, 8192, 16, "f16")])
def test_unequal_ranges_of_eight_waves(pkg, oracle, gpu, K, N, M, dtype):
    """Two chunks a wave and more, with and without left-over ones: the older waves of a workgroup take the longer ranges.  Each row of x meets
    one row of the weights, so that a range left out or met twice shows in every column."""
    pk, w = _weight(pkg, oracle, gpu, "gptq", K, N, 128, K + M, dtype)
    bf = dtype == "bf16"
    w = torch.from_numpy(oracle.to_f32(w, dtype) if bf else w.astype(np.float32)).to(gpu)
    for k0 in range(0, K, M * 61):
        ks = torch.arange(M, device=gpu) * 61 % K + k0
        ks = ks[ks < K]
        x = torch.zeros((M, K), dtype=torch.bfloat16 if bf else torch.float16, device=gpu)
        x[torch.arange(len(ks), device=gpu), ks] = 1
        got = pkg.ops.linear(pk, x).float()[: len(ks)]
        assert bool(((got - w[ks]).abs() <= 2.0 ** (-7 if bf else -10) * w[ks].abs()).all())  # (one weight, rounded once or twice)


# (decompositions that are no power of two, or another tile than the plan of powers of two: three workgroups along K of 128- and of 64-column
# tiles, whole K ranges of four waves, an odd one out with ragged chunks)
@pytest.mark.parametrize("K,N,M,dtype,gated", [(8192, 10240, 16, "f16", False), (3584, 4608, 13, "bf16", False), (4096, 22016, 8, "f16", True), (3584, 37888, 13, "bf16", True),
                                               (9088, 6400, 10, "f16", False), (3584, 37888, 1, "f16", True), (4096, 22016, 2, "f16", True), (8960, 2304, 1, "bf16", True),
                                               (3584, 4608, 1, "bf16", False), (8192, 10240, 40, "bf16", False), (5504, 4736, 24, "f16", True)])
def test_any_number_of_splits(pkg, oracle, gpu, K, N, M, dtype, gated):
    pk, w = _weight(pkg, oracle, gpu, "gptq", K, N, 128, M, dtype)
    x = oracle.make_x(M, K, seed=M, dtype=dtype)
    xt = to_dev(x, gpu, bf16=dtype == "bf16")
    if gated:
        _, want = oracle.gate_up_forward(x, w, "silu", None, dtype)
        got, again = (pkg.ops.linear_gate_up(pk, xt, "silu") for _ in range(2))
        assert max_rel_err(to_f32(got), oracle.to_f32(want, dtype)) <= TOL_GATED[dtype]
    else:
        y32, _ = oracle.linear_forward(x, w, None, dtype)
        got, again = (pkg.ops.linear(pk, xt) for _ in range(2))
        assert max_rel_err(to_f32(got), y32) <= TOL[dtype]
    assert torch.equal(got, again)
