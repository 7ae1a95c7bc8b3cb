"""FC backward (``csrc/fc_bwd_input.hip``, ``csrc/fc_soft_bwd.hip``, ``csrc/fc_lut.hip``) against
float64 at the edges of its tiling: several blocks of inputs and passes of
rows, inputs of more references than a lane's list, an input heavy in one
pass only, widths off the vector loads, batches off the 2- and 4-sample
tiles, one and several tiles per workgroup."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -23

# IN, OUT, K, B, candidates
CASES = [
    (784, 200, 8, 1, "random"),
    (50, 3001, 8, 5, "random"),       # about 960 references an input; odd rows
    (20, 300, 4, 7, "random"),
    (130, 6000, 8, 6, "one"),         # two passes; input 3 heavy in the first only
    (10300, 700, 5, 3, "random"),     # two blocks of inputs
    (1000, 10300, 2, 66, "random"),   # three passes
    (4097, 64, 8, 130, "random"),     # rows off the quad loads
    (512, 1030, 8, 1100, "random"),   # several tiles a workgroup, rows ahead
    (2000, 100, 16, 33, "random"),
    (64, 64, 1, 4, "random"),
    (300, 90, 8, 9, "same"),          # every candidate input 0
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%d-%d-K%d-B%d-%s" % c)
def test_fc_backward_matches_float64(case):
    from silogic_amd import ops
    IN, OUT, K, B, kind = case
    gen = torch.Generator().manual_seed(3)
    cand = torch.randint(0, IN, (OUT, 2, K), generator=gen)
    if kind == "one":
        cand[:200, 0] = 3
    if kind == "same":
        cand[:] = 0
    w = torch.softmax(torch.randn(OUT, 2, K, generator=gen), 2)
    c = torch.randn(OUT, 4, generator=gen)
    x, gy = torch.rand(B, IN, generator=gen), torch.randn(B, OUT, generator=gen)
    cand, w, c, x, gy = (t.cuda() for t in (cand.int(), w, c, x, gy))
    got = ops.fc_soft_bwd(x, cand, w, c, ops.GATE16, 1.0, gy)
    again = ops.fc_soft_bwd(x, cand, w, c, ops.GATE16, 1.0, gy)
    w64, c64, g64 = w.double(), c.double(), gy.double()
    xg = x.double()[:, cand.long().reshape(-1)].view(B, OUT, 2, K)
    a, b = ((xg * w64).sum(3))[..., 0], ((xg * w64).sum(3))[..., 1]
    ga, gb = g64 * (c64[:, 1] + c64[:, 3] * b), g64 * (c64[:, 2] + c64[:, 3] * a)
    grads = torch.stack([ga, gb], 2)                                   # [B, OUT, 2]
    terms = (grads.unsqueeze(3) * w64).reshape(B, -1)
    gx = torch.zeros(B, IN, dtype=torch.float64, device="cuda").index_add_(
        1, cand.long().reshape(-1), terms)
    # an operand gradient's own rounding: (K + 4) operations on terms of at most
    # (|c1| + |c3|) |g|; a sum of n terms rounds n times
    size = (g64.abs().unsqueeze(2).unsqueeze(3) * w64 *
            (c64[:, 1:3].abs() + c64[:, 3:].abs()).view(1, OUT, 2, 1)).reshape(B, -1)
    mass = torch.zeros_like(gx).index_add_(1, cand.long().reshape(-1), size)
    count = torch.zeros(IN, dtype=torch.float64, device="cuda").index_add_(
        0, cand.long().reshape(-1), torch.ones(OUT * 2 * K, dtype=torch.float64, device="cuda"))
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1])
    bound = EPS * (count + K + 8) * mass + 1e-30
    assert ((got[0].double() - gx).abs() <= bound).all()
    gw = (grads.unsqueeze(3) * xg).sum(0)
    wmass = (grads.abs().unsqueeze(3) * xg + EPS).sum(0) + (g64.abs().unsqueeze(2).unsqueeze(3) * xg *
            (c64[:, 1:3].abs() + c64[:, 3:].abs()).view(1, OUT, 2, 1)).sum(0)
    assert ((got[1].double() - gw).abs() <= EPS * (B + K + 8) * wmass).all()
    gc = torch.stack([g64.sum(0), (g64 * a).sum(0), (g64 * b).sum(0), (g64 * a * b).sum(0)], 1)
    cmass = g64.abs().sum(0).unsqueeze(1)
    assert ((got[2].double() - gc).abs() <= EPS * (B + 2 * K + 8) * cmass).all()


@pytest.mark.parametrize("arity,IN,OUT,K,B", [(3, 77, 333, 4, 5), (6, 40, 1801, 8, 9),
                                              (4, 4000, 513, 8, 66)])
def test_fc_lut_input_gradient_matches_float64(arity, IN, OUT, K, B):
    from silogic_amd import ops
    gen = torch.Generator().manual_seed(4)
    cand = torch.randint(0, IN, (OUT, arity, K), generator=gen).int().cuda()
    w = torch.softmax(torch.randn(OUT, arity, K, generator=gen), 2).cuda()
    s = torch.rand(OUT, 2 ** arity, generator=gen).cuda()
    x, gy = torch.rand(B, IN, generator=gen).cuda(), torch.randn(B, OUT, generator=gen).cuda()
    gx = ops.fc_lut_soft_bwd(x, cand, w, s, gy, True, False, False)[0]
    x64 = x.double().requires_grad_(True)
    v = (x64[:, cand.long().reshape(-1)].view(B, OUT, arity, K) * w.double()).sum(3)
    t = s.double().expand(B, OUT, -1)
    for j in range(arity):
        t = t[..., 0::2] + v[..., j:j + 1] * (t[..., 1::2] - t[..., 0::2])
    want, = torch.autograd.grad(t[..., 0], x64, gy.double())
    # rounding of about refs + 3 arity operations against sums of mixed sign
    refs = OUT * arity * K / IN
    rel = ((gx.double() - want).norm() / want.norm()).item()
    assert rel < EPS * (refs ** 0.5 + 3 * arity + K), rel


@pytest.mark.parametrize("arity,OUT,K,B", [(2, 1, 1, 1), (3, 65, 4, 9), (4, 63, 8, 700), (6, 70, 5, 1300)])
def test_fc_lut_parameter_gradients_match_float64(arity, OUT, K, B):
    # partial sums over one range of samples, a few, more than a step of 64
    from silogic_amd import ops
    IN = 40
    gen = torch.Generator().manual_seed(5)
    cand = torch.randint(0, IN, (OUT, arity, K), generator=gen).int().cuda()
    w = torch.softmax(torch.randn(OUT, arity, K, generator=gen), 2).cuda()
    s = torch.rand(OUT, 2 ** arity, generator=gen).cuda()
    x, gy = torch.rand(B, IN, generator=gen).cuda(), torch.randn(B, OUT, generator=gen).cuda()
    _, gw, gs = ops.fc_lut_soft_bwd(x, cand, w, s, gy, False, True, True)
    w64, s64 = w.double().requires_grad_(True), s.double().requires_grad_(True)
    v = (x.double()[:, cand.long().reshape(-1)].view(B, OUT, arity, K) * w64).sum(3)
    t = s64.expand(B, OUT, -1)
    for j in range(arity):
        t = t[..., 0::2] + v[..., j:j + 1] * (t[..., 1::2] - t[..., 0::2])
    want = torch.autograd.grad(t[..., 0], (w64, s64), gy.double())
    # B terms of mixed sign, each after about 3 arity + K roundings
    for got, ref in ((gw, want[0]), (gs, want[1])):
        rel = ((got.double() - ref).norm() / ref.norm()).item()
        assert rel < EPS * (B ** 0.5 + 3 * arity + K), rel
