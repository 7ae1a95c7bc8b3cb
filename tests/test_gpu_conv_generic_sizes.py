"""The generic conv forward at the edges of its launch: several channels a workgroup
(whole batches against their samples one by one, which take one channel each: the
same bits), maps below and above a workgroup's 256 positions, and an image that
passes the 32-bit form, against the same expression in torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(kind, depth, arity, K, C, N, kernel, gen):
    from silogic_amd import ops
    leaves, nodes, P = ops.tree_shape(kind, depth, arity)
    cm = torch.randint(0, C, (N, leaves, K), generator=gen, dtype=torch.int32).cuda()
    ch, cw = (torch.randint(0, kernel, (N, leaves, K), generator=gen, dtype=torch.int32).cuda()
              for _ in range(2))
    w = torch.softmax(torch.randn(N, leaves, K, generator=gen), 2).cuda()
    return torch.randn(N, nodes, P, generator=gen).cuda(), w, cm, ch, cw


@pytest.mark.parametrize("pool", [False, True])
@pytest.mark.parametrize("node,depth,arity,K,C,H,W,N,B", [
    ("walsh", 1, 2, 1, 3, 9, 7, 130, 601),       # 63 positions, channels not a multiple of 4
    ("walsh", 2, 2, 2, 5, 16, 16, 67, 256),      # 256 positions: a sample a workgroup
    ("walsh", 1, 2, 4, 2, 33, 31, 41, 130),      # 1023 positions
    ("multilinear", 2, 2, 1, 4, 20, 13, 66, 300),
    ("walsh", 1, 2, 1, 2, 2, 2, 4099, 257),      # one pooled position a sample
])
def test_channels_of_a_workgroup(node, depth, arity, K, C, H, W, N, B, pool):
    from silogic_amd import ops
    gen = torch.Generator().manual_seed(5)
    kind = {"walsh": ops.WALSH, "multilinear": ops.MULTILINEAR2}[node]
    args = _layer(kind, depth, arity, K, C, N, 3, gen)
    x = torch.rand(B, C, H, W, generator=gen).cuda()
    with torch.no_grad():
        whole = ops.conv_soft(x, *args, kind, depth, arity, K, 1, pool)
        for b in (0, 1, B // 2, B - 2, B - 1):
            one = ops.conv_soft(x[b:b + 1].contiguous(), *args, kind, depth, arity, K, 1, pool)
            assert torch.equal(whole[b:b + 1], one)
        for b in range(0, B, 64):
            some = ops.conv_soft(x[b:b + 5].contiguous(), *args, kind, depth, arity, K, 1, pool)
            assert torch.equal(whole[b:b + 5], some)


@pytest.mark.parametrize("pool", [False, True])
def test_an_image_past_the_32_bit_form(pool):
    from silogic_amd import ops
    gen = torch.Generator().manual_seed(6)
    C, H, W = 33, 4095, 4095                # 2.2 GB a sample
    npar, w, cm, ch, cw = _layer(ops.WALSH, 1, 2, 1, C, 2, 3, gen)
    x = torch.rand(1, C, H, W, device="cuda", generator=torch.Generator("cuda").manual_seed(6))
    with torch.no_grad():
        got = ops.conv_soft(x, npar, w, cm, ch, cw, ops.WALSH, 1, 2, 1, 1, pool)
    for n in range(2):
        a, b = (torch.nn.functional.pad(x[0, cm[n, i, 0]], (1, 1, 1, 1))[
            ch[n, i, 0]:ch[n, i, 0] + H, cw[n, i, 0]:cw[n, i, 0] + W] for i in range(2))
        c = npar[n, 0]
        y = torch.sigmoid(c[0] + c[1] * a + c[2] * b + c[3] * a * b)
        if pool:
            y = torch.nn.functional.max_pool2d(y[None], 2)[0]
        assert (got[0, n] - y).abs().max().item() < 1e-6   # a few roundings of values below 1
