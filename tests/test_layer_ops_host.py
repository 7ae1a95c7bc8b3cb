"""The layers' choice of a training path and its operators' refusals, without a
GPU (meta tensors stand for sizes that no test allocates)."""
import pytest
import torch

import silogic_amd as sl
from silogic_amd import library, ops


@pytest.mark.parametrize("node,outs", [("gate16", 1 << 27), ("multilinear", 1 << 27)])
def test_candidates_past_the_backward_kernels_keep_the_composite_backward(monkeypatch, node, outs):
    # 2 * OUT * K = 2^31: slg_fc_soft_bwd refuses it, the torch expression does not
    monkeypatch.setattr(ops, "param_levels_ok", lambda *a: True)
    m = sl.LogicLayer(20, 30, node=node, k=8, seed=1)
    assert m._params_op(m.node.raw())
    cand = torch.empty((outs, 2, 8), device="meta", dtype=torch.int32)
    monkeypatch.setattr(m._conn, "candidates_i32", lambda: cand)
    assert not m._params_op(m.node.raw())


def test_a_backward_without_kernels_says_so(monkeypatch):
    monkeypatch.setattr(ops, "fc_soft_bwd", lambda *a: None)
    t = torch.zeros
    with pytest.raises(NotImplementedError, match="fc_layer backward"):
        library.fc_layer_bwd(t(1, 3), t(2, 2, 1, dtype=torch.int32), t(2, 2, 1), t(10, 4), ops.GATE16, 1.0,
                             t(1, 2), True, True, True)
