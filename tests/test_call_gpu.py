"""The eager call as one C function (csrc/bindings/q4_call.cpp) against the Python code it stands for."""

import pytest
import torch

from tests.util import to_dev

pytestmark = pytest.mark.gpu


def _weight(pkg, oracle, gpu, layout, K=512, N=512, gs=128):
    if layout == "awq":
        qw, qz, sc = oracle.make_awq(K, N, gs, seed=1)
        return pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), None, gs, 1)
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=1, sym=False, act_order=layout == "act")
    return pkg.ops.make_packed(to_dev(qw, gpu), to_dev(qz, gpu), to_dev(sc, gpu), to_dev(gi, gpu) if layout == "act" else None, gs, 0)


@pytest.mark.parametrize("layout", ["gptq", "awq", "act"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bytes(pkg, oracle, gpu, layout, dtype):
    pk = _weight(pkg, oracle, gpu, layout)
    gen = torch.Generator(device=gpu).manual_seed(5)
    for M in (1, 5, 32, 33, 100, 300):
        for bias in (None, torch.randn(512, device=gpu, generator=gen).to(dtype)):
            x = torch.randn((M, 512), device=gpu, generator=gen).to(dtype)
            want = pkg.ops.linear(pk, x, bias)  # leaves the plan and the stream's workspace behind
            got = pk.call()(x, bias)
            if layout == "act" and M >= pkg._lib.REGROUP_MIN_ROWS:
                assert got is None
            else:
                assert got.shape == want.shape and got.dtype == dtype and torch.equal(got, want)
                assert torch.equal(pk.call()(x.view(1, M, 512), bias), want.view(1, M, 512))
            assert torch.equal(pkg.ops.apply_linear(pk, x, bias), want)


def test_tuned_plan(pkg, oracle, gpu):
    pk = _weight(pkg, oracle, gpu, "gptq", K=2048, N=4096)
    x = torch.randn((1, 2048), device=gpu).half()
    path, need, _ = pk.plan(1, pkg._lib.DTYPE_F16)
    cfg = pkg.ops.decode_candidates(pk, 1)[-1]
    pk._plans[(1, pkg._lib.DTYPE_F16)] = (path, need, cfg)
    want = pkg.ops.linear(pk, x)
    got = pk.call()(x, None)
    assert torch.equal(got, want)


def test_other_forms_are_left_to_the_python_code(pkg, oracle, gpu):
    pk = _weight(pkg, oracle, gpu, "gptq")
    x = torch.randn((4, 512), device=gpu).half()
    want = pkg.ops.linear(pk, x)
    call = pk.call()
    assert torch.equal(call(x, None), want)
    storage = torch.empty(4 * 512 + 1, device=gpu, dtype=torch.float16)
    unaligned = storage[1:].view(4, 512).copy_(x)
    strided = torch.empty((4, 1024), device=gpu, dtype=torch.float16)[:, ::2].copy_(x)
    for other in (unaligned, strided, torch.nn.Parameter(x), x.clone().requires_grad_()):
        assert call(other, None) is None
        assert torch.equal(pkg.ops.apply_linear(pk, other, None), want)
    with torch.no_grad():
        assert torch.equal(call(x.clone().requires_grad_(), None), want)
    for other in (x[:0], x.float(), x.cpu(), x[:, :256].contiguous(), x[0]):
        assert call(other, None) is None
    assert call(x[:3].contiguous(), torch.ones(512, device=gpu)) is None  # a bias of another type
    with torch.overrides.TorchFunctionMode():
        assert call(x, None) is None
    pk._plans.clear()  # a row count not met before
    assert call(x, None) is None and not pk._plans
    assert torch.equal(call(x, None, pk), want) and (4, pkg._lib.DTYPE_F16) in pk._plans  # planned by the weight, run by the function
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # a stream without a workspace
        known = (x.device.index, side.cuda_stream) in pkg.ops._workspaces  # (torch hands out streams from a pool)
        assert (call(x, None) is None) == (not known)
        assert torch.equal(pkg.ops.apply_linear(pk, x, None), want)
        assert torch.equal(call(x, None), want)
    side.synchronize()


def test_without_the_extension_module(pkg, oracle, gpu, monkeypatch):
    """The same bytes from the steps in Python."""
    pk, x = _weight(pkg, oracle, gpu, "gptq"), torch.randn((2, 3, 512), device=gpu).half()
    want = pkg.ops.apply_linear(pk, x, None)
    monkeypatch.setattr(pkg._lib, "_call", False)
    bare = _weight(pkg, oracle, gpu, "gptq")
    assert bare.call()(x, None) is None and torch.equal(pkg.ops.apply_linear(bare, x, None), want)


def test_captured_call(pkg, oracle, gpu):
    pk = _weight(pkg, oracle, gpu, "gptq", K=4096)
    pk.prepare()
    x = torch.randn((7, 4096), device=gpu).half()
    want = pkg.ops.linear(pk, x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = pkg.ops.apply_linear(pk, x, None)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(pkg.ops.apply_linear(pk, x, None), want)
