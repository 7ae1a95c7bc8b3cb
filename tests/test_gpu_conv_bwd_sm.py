"""Conv tree backward on sample-minor images (``csrc/conv_sm.hip``) against
float64 autograd of the same expression, at the edges of its tiling: batches
around the 64-sample chunk and past one round of chunks, odd maps and rows in
unequal steps, every node kind, candidate counts off the compiled 4 and 8,
kernels 1-5, trees of more than two channels, no pooling."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _reference(x, npar, w, cm, ch, cw, node, depth, arity, kernel, pool):
    B, C, H, W = x.shape
    N, leaves, K = cm.shape
    u = F.unfold(x, kernel, padding=kernel // 2)
    flat = (cm.long() * kernel + ch.long()) * kernel + cw.long()
    g = u.index_select(1, flat.reshape(-1)).view(B, N, leaves, K, -1)
    v = (g * w[None, ..., None]).sum(3)                              # [B, N, leaves, L]
    if node in ("gate16", "walsh"):
        nb = 0
        while v.shape[2] > 1:
            m = v.shape[2] // 2
            c = npar[None, :, nb:nb + m, :, None]
            a, b = v[:, :, 0::2], v[:, :, 1::2]
            z = c[:, :, :, 0] + c[:, :, :, 1] * a + c[:, :, :, 2] * b + c[:, :, :, 3] * a * b
            v = torch.sigmoid(z) if node == "walsh" else z
            nb += m
        y = v[:, :, 0]
    else:
        def lut(t):
            s = npar.reshape(1, N, -1, 1)
            for j in range(arity):
                s = s[:, :, 0::2] + t[:, :, j:j + 1] * (s[:, :, 1::2] - s[:, :, 0::2])
            return s[:, :, 0]
        y = lut(v)
        if node == "hybrid":
            y = lut((v >= 0.5).double()).detach() + (y - y.detach())
    y = y.view(B, N, H, W)
    return F.max_pool2d(y, 2, 2) if pool else y


# node, depth, arity, K, C, H, W, N, kernel, n_chan, B, pool
CASES = [
    ("gate16", 2, 2, 4, 6, 14, 14, 10, 3, 2, 65, True),
    ("gate16", 1, 2, 1, 3, 8, 10, 5, 3, 2, 1, True),
    ("gate16", 2, 2, 8, 5, 9, 11, 7, 5, 2, 63, True),     # odd map, 5 outputs a row
    ("gate16", 3, 2, 8, 4, 8, 8, 6, 3, 2, 64, True),
    ("gate16", 3, 2, 3, 8, 6, 37, 5, 3, 5, 70, True),     # 18 outputs a row, 5 channels a tree
    ("gate16", 2, 2, 5, 2, 7, 7, 4, 1, 1, 130, True),     # kernel 1: no border
    ("walsh", 2, 2, 4, 3, 10, 18, 9, 3, 2, 66, True),     # 9 outputs: steps of 5 and 4
    ("walsh", 3, 2, 2, 3, 8, 8, 5, 3, 2, 12, True),
    ("walsh", 1, 2, 8, 3, 8, 8, 5, 5, 3, 64, False),
    ("multilinear", 1, 6, 4, 7, 8, 8, 9, 3, 2, 65, True),
    ("multilinear", 1, 5, 8, 3, 7, 9, 4, 3, 2, 64, True),
    ("multilinear", 1, 3, 2, 3, 8, 8, 4, 5, 3, 40, True),
    ("multilinear", 1, 2, 4, 3, 6, 5, 4, 3, 2, 64, False),
    ("hybrid", 1, 6, 8, 5, 8, 8, 5, 3, 2, 65, True),
    ("hybrid", 1, 4, 4, 5, 8, 12, 5, 3, 3, 64, True),
    ("gate16", 3, 2, 2, 3, 32, 32, 64, 3, 2, 530, True),  # two rounds of 64-sample chunks
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-d%d-a%d-K%d-%dx%dx%d-N%d-k%d-c%d-B%d-%d" % c)
def test_conv_backward_matches_float64(case):
    from silogic_amd import ops
    node, depth, arity, K, C, H, W, N, kernel, n_chan, B, pool = case
    kind = {"gate16": ops.GATE16, "walsh": ops.WALSH, "multilinear": ops.MULTILINEAR2,
            "hybrid": ops.HYBRID}[node]
    gen = torch.Generator().manual_seed(7)
    leaves, nodes, P = ops.tree_shape(kind, depth, arity)
    chans = torch.stack([torch.randperm(C, generator=gen)[:n_chan] for _ in range(N)])
    pick = torch.randint(0, chans.shape[1], (N, leaves, K), generator=gen)
    cm = torch.gather(chans.unsqueeze(1).expand(N, leaves, -1), 2, pick).int()
    ch = torch.randint(0, kernel, (N, leaves, K), generator=gen).int()
    cw = torch.randint(0, kernel, (N, leaves, K), generator=gen).int()
    w = torch.softmax(torch.randn(N, leaves, K, generator=gen), 2)
    npar = torch.rand(N, nodes, P, generator=gen) if node in ("multilinear", "hybrid") else \
        torch.randn(N, nodes, P, generator=gen)
    x = torch.rand(B, C, H, W, generator=gen)
    half = (H // 2, W // 2) if pool else (H, W)
    gy = torch.randn(B, N, *half, generator=gen)
    dev = "cuda"
    x, w, npar, cm, ch, cw, gy = (t.to(dev) for t in (x, w, npar, cm, ch, cw, gy))

    got = ops.conv_soft_bwd(x, npar, w, cm, ch, cw, kind, depth, arity, K, kernel // 2, pool, gy)
    again = ops.conv_soft_bwd(x, npar, w, cm, ch, cw, kind, depth, arity, K, kernel // 2, pool, gy)
    leaf = [t.double().requires_grad_(True) for t in (x, npar, w)]
    want = [torch.zeros_like(t) for t in leaf]
    for b in range(0, B, 32):
        y = _reference(leaf[0][b:b + 32], leaf[1], leaf[2], cm, ch, cw, node, depth, arity, kernel,
                       pool)
        g = torch.autograd.grad(y, leaf, gy[b:b + 32].double())
        want = [s + t for s, t in zip(want, g)]
    # fp32 sums of at most B * outputs terms and trees of at most 12 roundings;
    # one window routed the other way at a near-tie (rounding against float64)
    # moves one output's gradient: sqrt(2 / outputs) of the norm
    outputs = gy.numel()
    bound = 5e-6 + (2.0 * (1 + 2e-5 * outputs) / outputs) ** 0.5 * (outputs > 20000)
    for name, a, a2, r in zip(("gx", "gnp", "gw"), got, again, want):
        assert torch.equal(a, a2), f"{name}: not the same bits twice"
        rel = ((a.double() - r).norm() / r.norm()).item()
        assert rel < bound, f"{name}: relative error {rel:.2e} (bound {bound:.1e})"
    # without the input gradient the sums are the same bits
    _, gn, gw = ops.conv_soft_bwd(x, npar, w, cm, ch, cw, kind, depth, arity, K, kernel // 2, pool,
                                  gy, need_x=False)
    assert torch.equal(gn, got[1]) and torch.equal(gw, got[2])


@pytest.mark.parametrize("case", [
    ("gate16", 3, 2, 4, 2, 8, 8, 96, 5, 2, 65, True),       # lists in 16 parts, cut inside a leaf's taps
    ("multilinear", 1, 6, 4, 1, 6, 37, 40, 3, 1, 3, False),  # one channel
    ("walsh", 2, 2, 8, 3, 16, 16, 33, 3, 1, 130, True),     # a last chunk of two samples
], ids=lambda c: c[0])
def test_split_input_gradient_matches_float64(case):
    test_conv_backward_matches_float64(case)
