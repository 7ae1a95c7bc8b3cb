"""The layers' training operators (``slg_layer_params`` and its backward inside
``fc_layer``, ``fc_lut_layer``, ``conv_layer``) against the modules' torch
expressions of the same parameters, every node kind, wiring and depth."""
import pytest
import torch

import silogic_amd as sl
from silogic_amd import ops

pytestmark = pytest.mark.gpu

LAYERS = [("gate16", 2, "topk", 8, 1.0), ("gate16", 2, "fixed", 1, 1.0), ("gate16", 2, "topk", 16, 1.0),
          ("walsh", 2, "topk", 5, 0.5), ("multilinear", 2, "blocktopk", 8, 1.0),
          ("multilinear", 3, "topk", 4, 1.0), ("hybrid", 6, "topk", 8, 1.0),
          ("hybrid", 2, "topk", 1, 1.0)]
BLOCKS = [("gate16", 2, 1, "topk", 4, 1.0), ("gate16", 2, 2, "topk", 3, 1.0),
          ("gate16", 2, 3, "fixed", 1, 1.0), ("gate16", 2, 4, "topk", 2, 1.0),
          ("walsh", 2, 2, "topk", 4, 0.7), ("walsh", 2, 4, "topk", 2, 1.0),
          ("multilinear", 6, 1, "topk", 8, 1.0), ("multilinear", 3, 2, "topk", 2, 1.0),
          ("hybrid", 4, 1, "topk", 4, 1.0)]


def _both(monkeypatch, module, x, call, used):
    """Outputs and gradients on the operators and on the torch expressions."""
    got = []
    for on in (True, False):
        if not on:
            monkeypatch.setattr(ops, "param_levels_ok", lambda *a: False)
        x.grad = None
        module.zero_grad(set_to_none=True)
        y = call(x)
        assert (used in y.grad_fn.__class__.__name__ or used in str(y.grad_fn.name())) == on
        gy = torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).cuda()
        y.backward(gy)
        got.append([y.detach(), x.grad] + [p.grad for p in module.parameters()])
    return got


def _close(a, b):
    for s, t in zip(a, b):
        assert (s is None) == (t is None)
        if s is not None:
            # the two derive the parameters with a few fp32 roundings each
            # (softmax of 16, a product over 16): 32 eps of the tensor's norm
            assert (s - t).norm() <= 32 * 2.0 ** -23 * (t.norm() + 1e-6)


@pytest.mark.parametrize("node,arity,wiring,k,tau", LAYERS)
def test_fc_layers(monkeypatch, node, arity, wiring, k, tau):
    torch.manual_seed(0)
    m = sl.LogicLayer(37, 70, node=node, connectome=wiring, arity=arity, k=k, tau=tau, seed=1)
    m = m.cuda().train()
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(torch.randn(p.shape))
    x = torch.rand(9, 37).cuda().requires_grad_(True)
    lut = m.is_lut
    _close(*_both(monkeypatch, m, x, m, "fc_lut_layer" if lut else "fc_layer"))


@pytest.mark.parametrize("node,arity,depth,wiring,k,tau", BLOCKS)
def test_conv_blocks(monkeypatch, node, arity, depth, wiring, k, tau):
    torch.manual_seed(0)
    m = sl.ConvLogicTree(3, 5, tree_depth=depth, connect=wiring, k=k, node=node, arity=arity,
                         tau=tau, residual_init=False, seed=2).cuda().train()
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(torch.randn(p.shape))
    x = torch.rand(3, 3, 6, 8).cuda().requires_grad_(True)
    _close(*_both(monkeypatch, m, x, m.forward_pooled, "conv_layer"))


def test_conv_block_under_autocast_and_a_default_dtype(monkeypatch):
    # the kernels read 32-bit parameters: autocast's 16-bit basis product and a
    # 64-bit default's ones are converted first. The forward's parameters are
    # the same values on both paths; the gate gradients pass a bf16 product on
    # one side only: 2 roundings of 2^-8, of terms up to four times as large as
    # what p (d - p.d) leaves of them
    def both(wiring, k):
        torch.manual_seed(0)
        m = sl.ConvLogicTree(3, 5, connect=wiring, k=k, residual_init=False, seed=2).cuda().train()
        x = torch.rand(3, 3, 6, 8).cuda().requires_grad_(True)
        with monkeypatch.context() as mp:
            return _both(mp, m, x, m.forward_pooled, "conv_layer")

    with torch.autocast("cuda", dtype=torch.bfloat16):
        got, want = both("topk", 4)
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):
        assert (a - b).norm() <= 2.0 ** -5 * b.norm()
    m = sl.ConvLogicTree(3, 5, connect="fixed", residual_init=False, seed=2).cuda().train()
    x = torch.rand(3, 3, 6, 8).cuda()
    want = m.forward_pooled(x)
    torch.set_default_dtype(torch.float64)
    try:
        assert torch.equal(m.forward_pooled(x), want)
    finally:
        torch.set_default_dtype(torch.float32)


def test_frozen_parameters_and_input():
    torch.manual_seed(0)
    m = sl.LogicLayer(20, 30, k=4, seed=1).cuda().train()
    m.node.gate_logits.requires_grad_(False)
    x = torch.rand(5, 20).cuda()
    g, = torch.autograd.grad(m(x).sum(), [m._conn.conn])
    m.node.gate_logits.requires_grad_(True)
    g2, gl = torch.autograd.grad(m(x).sum(), [m._conn.conn, m.node.gate_logits])
    assert torch.equal(g, g2) and gl.shape == (30, 16)


def test_other_dtypes_and_transforms_keep_their_path():
    m = sl.LogicLayer(20, 30, k=4, seed=1).cuda().train()
    assert ops.param_levels_ok(m._conn.conn, [m.node.gate_logits], 4)
    assert not ops.param_levels_ok(m._conn.conn, [m.node.gate_logits.double()], 4)
    assert not ops.param_levels_ok(m._conn.conn.transpose(0, 2), [m.node.gate_logits], 4)
    assert not ops.param_levels_ok(None, [torch.empty(30 * 16 + 1).cuda()[1:].view(30, 16)], 4)
    seen = []
    torch.func.grad(lambda c: (seen.append(ops.param_levels_ok(c, [c], 4)), c.sum())[1])(
        torch.ones(4).cuda())
    assert seen == [False]


@pytest.mark.parametrize("node", ["gate16", "walsh"])
def test_operator_takes_parameters_at_any_offset(node):
    # a traced layer calls the operator whatever its parameters' addresses
    m = sl.LogicLayer(20, 30, node=node, k=4, seed=1).cuda().train()
    x = torch.rand(5, 20).cuda()
    got = []
    for off in (0, 1):
        raw = m.node.raw().detach()
        flat = torch.empty(raw.numel() + off, device="cuda")
        shifted = flat[off:].view(raw.shape).copy_(raw).requires_grad_(True)
        assert (shifted.data_ptr() % 16 == 0) == (off == 0)
        y = torch.ops.silogic_hip.fc_layer(x, m._conn.candidates_i32(), m._conn.conn, shifted,
                                           m.node.kind, 1.0)[0]
        got.append((y.detach(), torch.autograd.grad(y.sum(), shifted)[0]))
    assert all(torch.equal(a, b) for a, b in zip(*got))


def _modules():
    return [sl.LogicLayer(20, 30, node="gate16", k=4, seed=1),
            sl.LogicLayer(20, 30, node="walsh", k=4, seed=1),
            sl.LogicLayer(20, 30, node="hybrid", arity=3, k=4, seed=1),
            sl.ConvLogicTree(3, 5, node="gate16", k=4, seed=1),
            sl.ConvLogicTree(3, 5, node="walsh", k=4, seed=1),
            sl.ConvLogicTree(3, 5, node="multilinear", arity=4, k=4, seed=1)]


def _operator(m, x, conn, levels):
    """``m``'s training operator on other parameter tensors."""
    if isinstance(m, sl.ConvLogicTree):
        cm, ch, cw = m._taps()
        gate16 = m.node_name == "gate16"
        return torch.ops.silogic_hip.conv_layer(
            x, conn, *levels, *[None] * (5 - len(levels)), m.basis if gate16 else None, cm, ch, cw,
            m._kind(), m.d, m.node_arity, cm.shape[-1], m.padding, True,
            1.0 / m.tau if m.node_name == "walsh" else 1.0)[0]
    cand = m._conn.candidates_i32()
    if m.is_lut:
        return torch.ops.silogic_hip.fc_lut_layer(x, cand, conn, levels[0], bool(m.node.hybrid))[0]
    return torch.ops.silogic_hip.fc_layer(x, cand, conn, levels[0], m.node.kind, m._inv_tau())[0]


def _own(m):
    if isinstance(m, sl.ConvLogicTree):
        levels = list(m.gate_logits) if m.node_name == "gate16" else [n.raw() for n in m.tree_nodes]
        return m.conn, levels, torch.rand(3, 3, 6, 8)
    return m._conn.conn, [m.node.raw()], torch.rand(5, 20)


@pytest.mark.parametrize("i", range(6))
def test_operators_convert_other_layouts_and_types(i):
    m = _modules()[i].cuda().train()
    conn, levels, x = _own(m)
    conn, levels, x = conn.detach(), [t.detach() for t in levels], x.cuda()
    want = _operator(m, x, conn, levels)

    def strided(t):   # same values, outermost stride 1
        return t.movedim(0, -1).contiguous().movedim(-1, 0)

    for f in (strided, lambda t: t.double()):
        args = f(conn).requires_grad_(True), [f(t).requires_grad_(True) for t in levels]
        y = _operator(m, x, *args)
        assert torch.equal(y, want)
        plain = [conn.clone().requires_grad_(True)] + [t.clone().requires_grad_(True) for t in levels]
        gw = torch.autograd.grad(_operator(m, x, plain[0], plain[1:]).sum(), plain)
        for g, w, t in zip(torch.autograd.grad(y.sum(), [args[0], *args[1]]), gw, [args[0], *args[1]]):
            assert g.dtype == t.dtype and torch.equal(g.float(), w)


@pytest.mark.parametrize("i", range(6))
def test_operators_refuse_parameters_of_another_shape(i):
    # larger tensors: nothing is read past an end, whether or not it is refused
    m = _modules()[i].cuda().train()
    conn, levels, x = _own(m)
    conn, levels, x = conn.detach(), [t.detach() for t in levels], x.cuda()
    for bad in (torch.cat([conn, conn]), torch.cat([conn, conn], 2), conn.reshape(-1).repeat(2)):
        with pytest.raises((ValueError, IndexError, RuntimeError)):
            _operator(m, x, bad, levels)
    for bad in (torch.cat([levels[0]] * 2), torch.cat([levels[0]] * 2, -1)):
        with pytest.raises((ValueError, IndexError, RuntimeError)):
            _operator(m, x, conn, [bad, *levels[1:]])


def test_a_layer_with_a_replaced_connection_raises():
    m = sl.LogicLayer(20, 30, k=4, seed=1).cuda().train()
    m._conn.conn = torch.nn.Parameter(torch.randn(31, 2, 4, device="cuda"))
    with pytest.raises(ValueError):
        m(torch.rand(5, 20).cuda())


@pytest.mark.parametrize("data", [False, True], ids=["in-place", "data"])
@pytest.mark.parametrize("i", range(6))
def test_an_update_between_forward_and_backward(i, data):
    # the gradients are those of the parameters the forward ran with
    m = _modules()[i].cuda().train()
    conn, levels, x = _own(m)
    x = x.cuda().requires_grad_(True)
    call = m.forward_pooled if isinstance(m, sl.ConvLogicTree) else m
    leaves = [x, conn, *levels]
    y = call(x)
    gy = torch.randn(y.shape, generator=torch.Generator().manual_seed(2)).cuda()
    want = torch.autograd.grad(y, leaves, gy)
    y = call(x)
    with torch.no_grad():
        for p in (conn, *levels):
            (p.data if data else p).normal_()
    for got, ref in zip(torch.autograd.grad(y, leaves, gy), want):
        assert torch.equal(got, ref)


class _Drop(torch.autograd.Function):
    """Passes its input on and sends no gradient back."""

    @staticmethod
    def forward(ctx, y):
        return y.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("i", range(6))
def test_an_output_without_a_gradient_gives_zeros(monkeypatch, i):
    m = _modules()[i].cuda().train()
    conn, levels, x = _own(m)
    call = m.forward_pooled if isinstance(m, sl.ConvLogicTree) else m
    for on in (True, False):      # the operators, then the torch expressions
        if not on:
            monkeypatch.setattr(ops, "param_levels_ok", lambda *a: False)
        leaves = [x.cuda().requires_grad_(True), conn, *levels]
        grads = torch.autograd.grad(_Drop.apply(call(leaves[0])).sum(), leaves, allow_unused=True)
        for g, t in zip(grads, leaves):
            assert g is not None and g.shape == t.shape and not g.any()
