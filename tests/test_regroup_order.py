"""The row order an act-order weight regroups by follows its g_idx: entries written in place after it was
found (load_state_dict copies into the buffers) take the weight back to the kernels that read g_idx."""

from __future__ import annotations

import copy

import numpy as np
import torch


def test_order_follows_g_idx(pkg, oracle):
    K, N, gs, M, f16 = 1024, 16384, 128, 2048, 0
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=3, sym=False, act_order=True)
    t = [torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)) for a in (qw, qz, sc, gi)]
    pk = pkg.ops.make_packed(*t, gs, 0)
    pk.find_order()
    assert pk.regroup(M, f16, False) > 0
    assert copy.deepcopy(pk).regroup(M, f16, False) > 0

    other = pk.g_idx.roll(1)
    pk.g_idx.copy_(other)
    assert pk.regroup(M, f16, False) == 0
    assert copy.deepcopy(pk).regroup(M, f16, False) == 0

    pk.find_order()
    assert pk.regroup(M, f16, False) > 0
    assert torch.equal(pk.order.long(), torch.argsort(other.long(), stable=True))
    pk.g_idx.fill_(0)  # groups of other sizes: none
    pk.find_order()
    assert pk.order is None and pk.regroup(M, f16, False) == 0


def test_inference_tensors_have_no_order(pkg, oracle):
    qw, qz, sc, gi = oracle.make_gptq(256, 64, 64, seed=4, sym=False, act_order=True)
    with torch.inference_mode():
        t = [torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).clone() for a in (qw, qz, sc, gi)]
        pk = pkg.ops.make_packed(*t, 64, 0)
        pk.find_order()
    assert pk.order is None


def test_copies_made_under_inference_mode(pkg, oracle):
    """A serving process copies layers in that mode; the copy's tensors count no writes."""
    qw, qz, sc, gi = oracle.make_gptq(256, 64, 64, seed=5, sym=False, act_order=True)
    t = [torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)) for a in (qw, qz, sc, gi)]
    pk = pkg.ops.make_packed(*t, 64, 0)
    pk.find_order()
    with torch.inference_mode():
        new = copy.deepcopy(pk)
    assert torch.equal(new.g_idx, pk.g_idx) and new.regroup(2048, 0, False) == 0
