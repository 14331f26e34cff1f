"""Act-order weights regrouped inside the call (q4_linear_regroup): the copy's rows must be the
checkpoint's in group order, so a one-hot activation reads every weight back as the oracle
dequantizes it, and sums agree with the oracle within fp32-accumulation noise plus the final rounding
(rel 2^-11 fp16, 2^-8 bf16 of the largest entry, times four for the sum's order and cancellation)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def to_dev(a, gpu):
    a = a.view(np.int32) if a.dtype == np.uint32 else a
    return torch.from_numpy(np.ascontiguousarray(a)).to(gpu)


def build(pkg, oracle, gpu, K, N, gs, seed):
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=seed, sym=False, act_order=True)
    pk = pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), to_dev(gi, gpu), gs, 0)
    return (qw, qz, sc, gi), pk


def call(pkg, pk, x, act=-1):
    lib, L = pkg._lib.load(), pkg._lib
    M, code = x.shape[0], pkg.ops._DTYPES[x.dtype]
    need, room = ctypes.c_size_t(0), ctypes.c_size_t(0)
    L.check(lib.q4_linear_regroup_plan(ctypes.byref(pk.struct()), M, code, int(act >= 0), ctypes.byref(need), ctypes.byref(room)))
    assert room.value > 0
    ws = torch.zeros(need.value, dtype=torch.uint8, device=x.device)
    scratch = torch.full((room.value,), 0xA5, dtype=torch.uint8, device=x.device)
    y = torch.empty((M, pk.N // (2 if act >= 0 else 1)), dtype=x.dtype, device=x.device)
    args = [ctypes.byref(pk.struct()), x.data_ptr(), None, y.data_ptr(), M, code, act, ws.data_ptr(), need.value, scratch.data_ptr()]
    assert lib.q4_linear_regroup(*args, room.value - 1, pkg.ops._stream_handle(x.device)) == L.ERR_WORKSPACE
    L.check(lib.q4_linear_regroup(*args, room.value, pkg.ops._stream_handle(x.device)))
    return y


# panels of 32, 16 and 8 columns: one workgroup's panel per CU or fewer, K at the edge of each width
@pytest.mark.parametrize("K,N,gs,M", [
    (128, 64, 32, 130), (1024, 8192, 128, 17), (2048, 272, 64, 33), (9600, 8192, 128, 129), (9728, 8192, 128, 40),
    (19200, 256, 128, 64), (19328, 264, 128, 65), (38400, 136, 128, 20),
])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_regrouped_call_matches_oracle(pkg, oracle, gpu, K, N, gs, M, dtype):
    (qw, qz, sc, gi), pk = build(pkg, oracle, gpu, K, N, gs, seed=K + N)
    w = oracle.dequant_gptq(qw, qz, sc, gi, gs, dtype)
    wf = w.view(np.uint16).astype(np.uint32) if dtype == "bf16" else w
    wf = (wf << 16).view(np.float32) if dtype == "bf16" else wf.astype(np.float32)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    rng = np.random.default_rng(M)
    rows = rng.choice(K, size=min(M, K), replace=False)
    one = torch.zeros((M, K), dtype=tdt, device=gpu)
    one[torch.arange(len(rows)), torch.from_numpy(rows).to(gpu)] = 1
    got = call(pkg, pk, one).float().cpu().numpy()
    assert np.array_equal(got[:len(rows)], wf[rows])
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(gpu).to(tdt)
    got = call(pkg, pk, x).float().cpu().numpy()
    want = x.float().cpu().numpy() @ wf
    assert np.abs(got - want).max() <= 4 * (2.0 ** -8 if dtype == "bf16" else 2.0 ** -11) * np.abs(want).max()


@pytest.mark.parametrize("K,N,M,regroups", [(512, 32768, 48, False), (4096, 28672, 48, False), (8192, 32768, 48, False), (8256, 33024, 48, True), (4096, 28672, 130, True), (4096, 4096, 1024, False), (4096, 6144, 1536, True),
                                          (14336, 4096, 301, True), (14336, 4096, 400, False), (4096, 6144, 700, True), (3584, 4608, 1100, True)])
def test_layers_regroup_from_the_librarys_row_count_on(pkg, oracle, gpu, K, N, M, regroups):
    """The tensor calls take the regrouped route by the library's rule; gated and plain agree with the
    kernels that read through g_idx (the same weights, sums in another order)."""
    _, pk = build(pkg, oracle, gpu, K, N, 64 if K % 128 else 128, seed=N)
    x = torch.randn((M, K), device=gpu, dtype=torch.float16) * 0.1
    assert (pk.regroup(M, 0, False)[1] > 0) == regroups
    plain = pkg.ops.linear(pk, x, path=2)
    for a, b in ((pkg.ops.linear(pk, x), plain), (pkg.ops.linear_gate_up(pk, x), pkg.ops.act_mul(plain))):
        assert ((a.float() - b.float()).norm() / b.float().norm()).item() <= 2e-3
    assert pkg.ops.linear(pk, x[:0]).shape == (0, N)


# On the size below the library regroups from 129 rows on: just above, and well inside
ROWS = [130, 200]


def big(pkg, gpu, seed):
    K, N, gs = 8192, 32768, 128
    gen = torch.Generator(device=gpu).manual_seed(seed)
    words = lambda *s: torch.randint(-(2**31), 2**31 - 1, s, dtype=torch.int32, device=gpu, generator=gen)  # noqa: E731
    scales = (torch.rand((K // gs, N), device=gpu, generator=gen) * 0.019 + 0.001).half()
    g_idx = (torch.arange(K, device=gpu) // gs)[torch.randperm(K, device=gpu, generator=gen)].int()
    return pkg.ops.make_packed(words(K // 8, N), words(K // gs, N // 8), scales, g_idx, gs, 0)


def against_g_idx(pkg, pk, x, plain=None, gated=None):
    """Both calls against the kernels that read g_idx as it is in memory now."""
    want = pkg.ops.linear(pk, x, path=2)
    plain = pkg.ops.linear(pk, x) if plain is None else plain
    gated = pkg.ops.linear_gate_up(pk, x) if gated is None else gated
    for a, b in ((plain, want), (gated, pkg.ops.act_mul(want))):
        assert ((a.float() - b.float()).norm() / b.float().norm()).item() <= 2e-3


@pytest.mark.parametrize("M", ROWS)
def test_a_call_reads_g_idx_when_it_runs(pkg, gpu, M):
    """Entries written after the layer was prepared, counted by torch (copy_) or not (.data), are the ones used."""
    pk = big(pkg, gpu, M)
    pk.prepare()
    assert pk.regroup(M, 0, False)[1] > 0 and pk.regroup(M, 0, True)[1] > 0
    x = torch.randn((M, pk.K), device=gpu, dtype=torch.float16) * 0.1
    against_g_idx(pkg, pk, x)
    pk.g_idx.data.copy_(pk.g_idx[torch.randperm(pk.K, device=gpu)])
    against_g_idx(pkg, pk, x)
    pk.g_idx.copy_(pk.g_idx.flip(0))
    against_g_idx(pkg, pk, x)


@pytest.mark.parametrize("M", ROWS)
def test_a_captured_call_reads_g_idx_when_it_is_replayed(pkg, gpu, M):
    """Another checkpoint is copied into the buffers of a captured layer, as load_state_dict does it."""
    pk = big(pkg, gpu, M)
    pk.prepare()
    x = torch.randn((M, pk.K), device=gpu, dtype=torch.float16) * 0.1
    pkg.ops.linear(pk, x), pkg.ops.linear_gate_up(pk, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plain, gated = pkg.ops.linear(pk, x), pkg.ops.linear_gate_up(pk, x)
    for seed in range(3):
        src = big(pkg, gpu, seed)
        for name in ("qweight", "qzeros", "scales", "g_idx"):
            getattr(pk, name).copy_(getattr(src, name))
        pk.prepare()
        graph.replay()
        torch.cuda.synchronize()
        against_g_idx(pkg, pk, x, plain, gated)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_uneven_groups_are_looked_up(pkg, gpu, M, dtype):
    """Groups of other sizes, which only the device sees: the very kernels that read through g_idx."""
    pk = big(pkg, gpu, M)
    x = (torch.randn((M, pk.K), device=gpu) * 0.1).to(dtype)
    for entries in (pk.g_idx.clamp(max=pk.num_groups - 2), torch.zeros_like(pk.g_idx), pk.g_idx - 1, pk.g_idx + 1):
        pk.g_idx.copy_(entries)
        want = pkg.ops.linear(pk, x, path=2)
        assert torch.equal(pkg.ops.linear(pk, x), want)
        assert torch.equal(pkg.ops.linear_gate_up(pk, x), pkg.ops.act_mul(want))


@pytest.mark.parametrize("K,N,gs,M", [(128, 64, 32, 130), (2048, 272, 64, 33), (38400, 136, 128, 20), (1024, 8192, 1024, 64)])
def test_uneven_groups_without_a_prefill_kernel(pkg, oracle, gpu, K, N, gs, M):
    """Sizes that the library never regroups by itself, one group and columns in no whole tile among them."""
    _, pk = build(pkg, oracle, gpu, K, N, gs, seed=K)
    x = torch.randn((M, K), device=gpu, dtype=torch.float16) * 0.1
    pk.g_idx.copy_(pk.g_idx.clamp(max=pk.num_groups // 2 - 1) if pk.num_groups > 1 else pk.g_idx - 1)
    want = pkg.ops.linear(pk, x, path=2 if N % 128 == 0 else 3)
    assert torch.equal(call(pkg, pk, x), want)


def test_the_copy_lasts_for_one_call(pkg, gpu, monkeypatch):
    """Preparing a layer and calling it leaves no copy of the weight behind; without memory for one, or with `out` under
    capture, where nothing may be allocated, the call goes through g_idx."""
    pk = big(pkg, gpu, 1)
    x = torch.randn((200, pk.K), device=gpu, dtype=torch.float16) * 0.1
    pkg.ops.linear(pk, x[:1]), pkg.ops.linear(pk, x, path=2)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    pk.prepare(rows=(1, 48, 200))
    got = pkg.ops.linear(pk, x), pkg.ops.linear_gate_up(pk, x)
    kept = sum(t.numel() * t.element_size() for t in got)
    assert torch.cuda.memory_allocated() - before - kept < pk.K * pk.N // 2
    want = pkg.ops.linear(pk, x, path=2)
    out = torch.empty_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = torch.cuda.memory_allocated()
        pkg.ops.linear(pk, x, out=out)
        assert torch.cuda.memory_allocated() == held
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    empty = torch.empty

    def full(*args, **kwargs):
        if kwargs.get("dtype") == torch.uint8:
            raise torch.cuda.OutOfMemoryError("no memory for the copy")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", full)
    assert torch.equal(pkg.ops.linear(pk, x), want) and torch.equal(pkg.ops.linear_gate_up(pk, x), pkg.ops.act_mul(want))
