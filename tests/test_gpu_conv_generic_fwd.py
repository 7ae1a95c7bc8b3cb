"""Forward of the generic node trees where its lanes cross samples: maps of
one position, runs that end inside a sample, more samples than lanes, trees
held for four window positions at once (at most 16 leaves) and one at a time,
against the reference expressions. A leaf adds K = 4 products of weights that
sum to 1 and a level is a few roundings of values in [0, 1] or walsh
coefficients of order 1, so 1e-5 relative covers five levels (5 * ~10 ulp of
2^-24 = 3e-6); a hybrid value is a table entry.
"""
import pytest
import torch

import silogic_amd as sl
from oracle import torch_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("node,arity,depth,C,H,N,B", [
    ("walsh", 2, 2, 3, 2, 7, 600),    # one pooled position a sample
    ("walsh", 2, 2, 3, 14, 5, 21),    # 49 positions: runs end inside samples
    ("walsh", 2, 4, 4, 8, 3, 33),     # 16 leaves: four trees at once
    ("walsh", 2, 5, 4, 9, 3, 9),      # 32 leaves: one at a time; odd map
    ("multilinear", 3, 2, 3, 5, 1, 65),
    ("hybrid", 4, 2, 3, 32, 2, 1),    # 256 pooled positions exactly
])
def test_runs_across_samples(node, arity, depth, C, H, N, B):
    conv = sl.ConvLogicTree(C, N, kernel=3, tree_depth=depth, connect="topk", k=4, n_chan=2,
                            residual_init=False, seed=depth, node=node, arity=arity, tau=0.7)
    sd = {k: v.clone() for k, v in conv.state_dict().items()}
    blk = dict(prefix="", cin=C, n=N, kernel=3, depth=depth, stride=1, padding=conv.padding,
               connect="topk", k=4, node=node, node_arity=arity, leaves=conv.leaves, tau=0.7, hw=H)
    x = torch.rand(B, C, H, H, generator=torch.Generator().manual_seed(B))
    ref = torch_ref.conv_soft(blk, sd, x)
    conv = conv.to("cuda").eval()
    with torch.no_grad():
        y, yp = conv(x.cuda()).cpu(), conv.forward_pooled(x.cuda()).cpu()
    for got, want in ((y, ref), (yp, torch_ref.orpool_soft(ref))):
        assert got.shape == want.shape
        assert ((got - want).abs() <= 1e-5 * want.abs() + 1e-6).all(), (got - want).abs().max()
