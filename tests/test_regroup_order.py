"""Nothing read from an act-order weight's g_idx is kept with the weight: copies are made in every mode, and the
rule by which calls regroup looks at sizes only."""

from __future__ import annotations

import copy

import numpy as np
import pytest
import torch


def _packed(pkg, oracle, K, N, gs):
    qw, qz, sc, gi = oracle.make_gptq(K, N, gs, seed=3, sym=False, act_order=True)
    t = [torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)) for a in (qw, qz, sc, gi)]
    return pkg.ops.make_packed(*t, gs, 0)


def test_the_rule_looks_at_sizes_only(pkg, oracle):
    pk = _packed(pkg, oracle, 1024, 16384, 128)
    need = pk.regroup(4096, 0, False)
    assert min(need) > 0 and pk.regroup(32, 0, False) == (0, 0)
    other = copy.deepcopy(pk)
    other._plans.clear()
    other.g_idx.data.fill_(0)
    assert other.regroup(4096, 0, False) == need


@pytest.mark.parametrize("gate_up", [False, True])
def test_no_plan_keeps_room_for_the_copy(pkg, oracle, gate_up):
    """The workspace, which is kept and grown by doubling, holds partial sums only; the scratch, which lasts for one
    call, holds the weight, x and the row order, or a gated call's sums where they are larger."""
    K, N, M = 1024, 16384, 4096
    pk = _packed(pkg, oracle, K, N, 128)
    need, scratch = pk.regroup(M, 0, gate_up)
    contiguous = pkg.ops.make_packed(pk.qweight, pk.qzeros, pk.scales, None, 128, 0)
    assert pk.plan(M, 0)[1] == need
    own = pkg._lib.load().q4_workspace_bytes_for(pk.struct(), M)
    assert need == max(own, contiguous.plan(M, 0)[1])
    copy = max(K * N // 2, 2 * M * N if gate_up else 0)
    assert 0 <= scratch - (copy + 2 * M * K + 4 * K) <= 2048


@pytest.mark.parametrize("mode", [torch.inference_mode, torch.no_grad, torch.enable_grad])
def test_copies_in_every_mode(pkg, oracle, mode):
    """A serving process copies layers under inference_mode, where the copy's tensors count no writes."""
    pk = _packed(pkg, oracle, 1024, 16384, 128)
    with mode():
        new = copy.deepcopy(pk)
    assert torch.equal(new.g_idx, pk.g_idx) and new.regroup(4096, 0, False) == pk.regroup(4096, 0, False)
