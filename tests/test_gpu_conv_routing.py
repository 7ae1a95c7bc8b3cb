"""The pooled conv backward sends each gradient to the window position that its
forward's maximum came from: values in eighths and parameters in sevenths, where
rounding makes near-ties common, every tree, on images that fit LDS and larger ones.
The unpooled backward, fed the gradients at the forward's own first maxima, has
the same sums in another order."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SMALL, LARGE = (6, 16, 16), (44, 32, 32)
# node, depth, arity, K, (C, H, W), N, B
CASES = [
    ("walsh", 1, 2, 4, SMALL, 32, 192),
    ("walsh", 2, 2, 4, SMALL, 32, 192),
    ("walsh", 3, 2, 8, SMALL, 32, 192),
    ("walsh", 4, 2, 2, SMALL, 16, 64),     # deeper: the kernels with lanes along positions
    ("walsh", 2, 2, 4, LARGE, 16, 70),
    ("gate16", 1, 2, 4, SMALL, 32, 192),
    ("gate16", 2, 2, 4, SMALL, 32, 192),
    ("gate16", 3, 2, 4, SMALL, 32, 192),
    ("gate16", 4, 2, 2, SMALL, 16, 64),    # forward on LDS, backward through the caches
    ("gate16", 5, 2, 2, SMALL, 16, 64),
    ("gate16", 2, 2, 4, LARGE, 16, 70),
    ("gate16", 3, 2, 8, LARGE, 16, 70),
    ("multilinear", 1, 2, 4, SMALL, 32, 192),
    ("multilinear", 1, 4, 4, SMALL, 32, 192),
    ("multilinear", 1, 6, 4, SMALL, 32, 192),
    ("multilinear", 2, 3, 2, SMALL, 16, 64),
    ("multilinear", 1, 3, 4, LARGE, 16, 70),
    ("multilinear", 1, 4, 8, LARGE, 16, 70),
    ("multilinear", 1, 6, 4, LARGE, 16, 70),
    ("hybrid", 1, 6, 4, SMALL, 32, 192),
    ("hybrid", 1, 4, 4, LARGE, 16, 70),
]


def first_maximum(y):
    """Window positions (0-3, row-major) of the first maxima of ``y`` [B,N,H,W]."""
    B, N, H, W = y.shape
    win = y[:, :, :H // 2 * 2, :W // 2 * 2].reshape(B, N, H // 2, 2, W // 2, 2)
    win = win.permute(0, 1, 2, 4, 3, 5).reshape(B, N, H // 2, W // 2, 4)
    pos = torch.full(win.shape[:4], 3, device=y.device)
    for q in (2, 1, 0):
        pos = torch.where(win[..., q] == win.amax(-1), q, pos)
    return pos, win.amax(-1)


@pytest.mark.parametrize("weights", ["eighths", "softmax"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-d%d-a%d-K%d-%s-N%d-B%d" % (
    *c[:4], "lds" if c[4] is SMALL else "large", *c[5:]))
def test_pooled_backward_routes_on_the_forwards_values(case, weights):
    from silogic_amd import ops
    node, depth, arity, K, (C, H, W), N, B = case
    kind = {"gate16": ops.GATE16, "walsh": ops.WALSH, "multilinear": ops.MULTILINEAR2,
            "hybrid": ops.HYBRID}[node]
    gen = torch.Generator().manual_seed(11)
    leaves, nodes, P = ops.tree_shape(kind, depth, arity)
    chans = torch.stack([torch.randperm(C, generator=gen)[:2] for _ in range(N)])
    pick = torch.randint(0, 2, (N, leaves, K), generator=gen)
    cm = torch.gather(chans.unsqueeze(1).expand(N, leaves, -1), 2, pick).int()
    ch = torch.randint(0, 3, (N, leaves, K), generator=gen).int()
    cw = torch.randint(0, 3, (N, leaves, K), generator=gen).int()
    if weights == "eighths":
        w = torch.zeros(N, leaves, K).scatter_add_(
            2, torch.randint(0, K, (N, leaves, 8), generator=gen), torch.full((N, leaves, 8), 0.125))
    else:
        w = torch.softmax(torch.randn(N, leaves, K, generator=gen), 2)
    span = (0, 9) if node in ("multilinear", "hybrid") else (-8, 9)
    npar = torch.randint(*span, (N, nodes, P), generator=gen) / 7.0
    x = torch.randint(0, 9, (B, C, H, W), generator=gen) / 8.0
    gy = torch.randn(B, N, H // 2, W // 2, generator=gen)
    x, w, npar, cm, ch, cw, gy = (t.cuda() for t in (x, w, npar, cm, ch, cw, gy))
    args = (npar, w, cm, ch, cw, kind, depth, arity, K, 1)
    assert ops.conv_fits_lds((C, H, W), 1, True, kind, depth, arity, K) == \
        ops.conv_fits_lds((C, H, W), 1, False, kind, depth, arity, K)

    pos, top = first_maximum(ops.conv_soft(x, *args, False))
    assert torch.equal(ops.conv_soft(x, *args, True), top)
    sent = torch.zeros(B, N, H // 2, W // 2, 4, device="cuda").scatter_(4, pos.unsqueeze(4),
                                                                       gy.unsqueeze(4))
    sent = sent.view(B, N, H // 2, W // 2, 2, 2).permute(0, 1, 2, 4, 3, 5).reshape(B, N, H, W)
    got = ops.conv_soft_bwd(x, *args, True, gy)
    want = ops.conv_soft_bwd(x, *args, False, sent.contiguous())
    # the same terms summed in another order: 5e-6 as against float64; one window
    # of M sent elsewhere moves about sqrt(2 / M) of the norm, 2e-3 at least
    for name, a, b in zip(("gx", "gnp", "gw"), got, want):
        rel = ((a.double() - b.double()).norm() / b.double().norm()).item()
        assert rel < 5e-6, f"{name}: {rel:.2e}"
