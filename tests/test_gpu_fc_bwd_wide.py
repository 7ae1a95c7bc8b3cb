"""The FC input gradient of wide layers, gathered from sample-minor rows in memory,
against float64: more input blocks and passes than the way through LDS is worth, and
layers past its table. Inputs without references, odd widths, repeated candidates."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _sums(x, cand, w, gy, npar):
    """float64 operand gradients of gate16 nodes scattered to the inputs."""
    x, w, gy, p = (t.double() for t in (x, w, gy, npar))
    i = cand.long()
    a = (x[:, i[:, 0]] * w[:, 0]).sum(-1)
    b = (x[:, i[:, 1]] * w[:, 1]).sum(-1)
    ga, gb = gy * (p[:, 1] + p[:, 3] * b), gy * (p[:, 2] + p[:, 3] * a)
    gx = torch.zeros_like(x)
    for side, g in ((0, ga), (1, gb)):
        for k in range(cand.shape[2]):
            gx.index_add_(1, i[:, side, k], g * w[:, side, k])
    return gx


@pytest.mark.parametrize("B,IN,OUT,K", [
    (3, 70001, 33333, 2),
    (70, 24904, 24904, 2),
    (257, 16001, 15999, 1),
    (1, 1300000, 1300000, 2),     # its table passes 2^31 entries on the way through LDS
])
def test_wide_input_gradient_matches_float64(B, IN, OUT, K):
    from silogic_amd import ops
    gen = torch.Generator().manual_seed(3)
    x = torch.rand(B, IN, generator=gen).cuda()
    cand = torch.randint(0, IN, (OUT, 2, K), generator=gen, dtype=torch.int32).cuda()
    w = torch.softmax(torch.randn(OUT, 2, K, generator=gen), -1).cuda()
    npar, gy = torch.randn(OUT, 4, generator=gen).cuda(), torch.randn(B, OUT, generator=gen).cuda()
    got = ops.fc_soft_bwd(x, cand, w, npar, ops.GATE16, 1.0, gy)
    again = ops.fc_soft_bwd(x, cand, w, npar, ops.GATE16, 1.0, gy)
    want = _sums(x, cand, w, gy, npar)
    # fp32 operands of K terms and sums of a few references: a handful of roundings
    assert ((got[0].double() - want).norm() / want.norm()).item() < 1e-6
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_wide_lut_input_gradient_matches_float64():
    from silogic_amd import ops
    B, IN, OUT, A, K = 5, 36001, 30001, 3, 2
    gen = torch.Generator().manual_seed(4)
    x = torch.rand(B, IN, generator=gen).cuda().double().requires_grad_(True)
    cand = torch.randint(0, IN, (OUT, A, K), generator=gen, dtype=torch.int32).cuda()
    w = torch.softmax(torch.randn(OUT, A, K, generator=gen), -1).cuda()
    s, gy = torch.rand(OUT, 2 ** A, generator=gen).cuda(), torch.randn(B, OUT, generator=gen).cuda()
    v = (x[:, cand.long().reshape(-1)].view(B, OUT, A, K) * w.double()).sum(-1)
    t = s.double().unsqueeze(0)
    for j in range(A):
        t = t[..., 0::2] + v[:, :, j:j + 1] * (t[..., 1::2] - t[..., 0::2])
    want, = torch.autograd.grad(t[..., 0], x, gy.double())
    gx, _, _ = ops.fc_lut_soft_bwd(x.detach().float(), cand, w, s, gy)
    assert ((gx.double() - want).norm() / want.norm()).item() < 1e-6
