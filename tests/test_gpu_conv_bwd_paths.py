"""The conv backward's three sets of kernels at the same sizes: lanes along samples,
along output positions and the generic ones, each named by the caller, against
float64 and against the forward's own window positions. (Left to itself the
library takes one by size: ``test_conv_bwd_choice.py``.)"""
import functools

import pytest
from test_gpu_conv_bwd_sm import CASES, test_conv_backward_matches_float64 as _float64
from test_gpu_conv_routing import CASES as ROUTES
from test_gpu_conv_routing import test_pooled_backward_routes_on_the_forwards_values as _routes

pytestmark = pytest.mark.gpu

SAMPLES, POSITIONS, GENERIC = 1, 2, 3

# split reference lists, one channel, a last chunk of two samples
EXTRA = [
    ("gate16", 3, 2, 4, 2, 8, 8, 96, 5, 2, 65, True),
    ("multilinear", 1, 6, 4, 1, 6, 37, 40, 3, 1, 3, False),
    ("walsh", 2, 2, 8, 3, 16, 16, 33, 3, 1, 130, True),
    ("hybrid", 1, 2, 1, 3, 9, 7, 5, 3, 2, 1, False),
    ("gate16", 2, 2, 4, 40, 34, 34, 6, 3, 2, 2, True),    # an image past LDS
]


def _takes(path, node, depth):
    if path == GENERIC:
        return True
    binary = node in ("gate16", "walsh")
    return depth <= (3 if binary else 1) and not (path == POSITIONS and node == "walsh")


def _on(monkeypatch, path):
    from silogic_amd import ops
    monkeypatch.setattr(ops, "conv_soft_bwd", functools.partial(ops.conv_soft_bwd, path=path))


@pytest.mark.parametrize("case,path", [(c, p) for c in CASES + EXTRA for p in (SAMPLES, POSITIONS, GENERIC)
                                       if _takes(p, c[0], c[1])],
                         ids=lambda v: v if isinstance(v, int) else "%s-d%d-a%d-K%d-%dx%dx%d-N%d-k%d-c%d-B%d-%d" % v)
def test_paths_match_float64(case, path, monkeypatch):
    _on(monkeypatch, path)
    _float64(case)


@pytest.mark.parametrize("case,path", [(c, p) for c in ROUTES for p in (SAMPLES, POSITIONS, GENERIC)
                                       if _takes(p, c[0], c[1])],
                         ids=lambda v: v if isinstance(v, int) else "%s-d%d-a%d-K%d-%dx%dx%d-N%d-B%d" % (
                             *v[:4], *v[4], *v[5:]))
def test_paths_route_on_the_forwards_values(case, path, monkeypatch):
    _on(monkeypatch, path)
    _routes(case, "eighths")
