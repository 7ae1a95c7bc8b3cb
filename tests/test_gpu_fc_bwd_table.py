"""Input-gradient table of the FC backward built in one launch
(``ig_table_kernel``) and the general way, at the edges of the rule between
them and inside it: references in all, a block and an input, one and several
blocks, lists past a lane's, empty blocks, candidates out of range
(clamped), against float64. An input's sum of n terms rounds n times and a
term at most K + 8 times, so n + K + 8 units of its terms' mass bound it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -23

# IN, OUT, K, B, candidates
CASES = [
    (1000, 1000, 8, 256, "random"),    # 16000 references in 4 blocks
    (3072, 3072, 8, 5, "random"),      # 48K references: the most
    (3072, 3073, 8, 5, "random"),      # past them: the general way
    (300, 256, 8, 1030, "random"),     # 4096 references in one block
    (300, 257, 8, 1030, "random"),     # past them: the general way
    (64, 128, 8, 9, "random"),         # 32 references an input exactly
    (63, 128, 8, 9, "random"),         # more: the general way
    (3000, 1500, 8, 4, "first"),       # input 0 alone: 24000 references, empty blocks
    (3000, 250, 8, 1030, "last"),      # one block
    (9000, 3, 1, 1, "random"),         # nearly every list empty
    (700, 333, 3, 6, "outside"),       # clamped
    (1, 2, 8, 3, "random"),            # one input, 32 references
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%d-%d-K%d-B%d-%s" % c)
def test_input_gradient_table(case):
    from silogic_amd import ops
    IN, OUT, K, B, kind = case
    gen = torch.Generator().manual_seed(5)
    cand = torch.randint(0, IN, (OUT, 2, K), generator=gen)
    if kind == "first":
        cand[:] = 0
    if kind == "last":
        cand[:] = IN - 1
    if kind == "outside":
        cand[::3] = IN + 5
        cand[1::3] = -2
    used = cand.clamp(0, IN - 1).reshape(-1).cuda()
    w = torch.softmax(torch.randn(OUT, 2, K, generator=gen), 2)
    c = torch.randn(OUT, 4, generator=gen)
    x, gy = torch.rand(B, IN, generator=gen), torch.randn(B, OUT, generator=gen)
    cand, w, c, x, gy = (t.cuda() for t in (cand.int(), w, c, x, gy))
    got = ops.fc_soft_bwd(x, cand, w, c, ops.GATE16, 1.0, gy)[0]
    again = ops.fc_soft_bwd(x, cand, w, c, ops.GATE16, 1.0, gy)[0]
    assert torch.equal(got, again)
    w64, c64, g64 = w.double(), c.double(), gy.double()
    v = (x.double()[:, used].view(B, OUT, 2, K) * w64).sum(3)
    grads = torch.stack([g64 * (c64[:, 1] + c64[:, 3] * v[..., 1]),
                         g64 * (c64[:, 2] + c64[:, 3] * v[..., 0])], 2)
    scatter = lambda t: torch.zeros(B, IN, dtype=torch.float64, device="cuda").index_add_(
        1, used, t.reshape(B, -1))
    want = scatter(grads.unsqueeze(3) * w64)
    mass = scatter(g64.abs().unsqueeze(2).unsqueeze(3) * w64 *
                   (c64[:, 1:3].abs() + c64[:, 3:].abs()).view(1, OUT, 2, 1))
    count = torch.bincount(used, minlength=IN).double()
    assert ((got.double() - want).abs() <= EPS * (count + K + 8) * mass + 1e-30).all()
