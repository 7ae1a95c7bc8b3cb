"""Which kernels the conv backward takes, and its workspace: the kernels with lanes along samples where there are samples enough, the others for few of
them, as measured (``csrc/conv_bwd.hip``)."""
import pytest

from silogic_amd import _lib, ops

AUTO, SAMPLES, POSITIONS, GENERIC = range(4)
pytestmark = pytest.mark.skipif(not _lib.available(), reason="library not built")


def _floats(path, B, C, H, N, kind, depth, arity, K, pad, pool, want_gx=1):
    return _lib.lib().slg_conv_soft_bwd_workspace_on(path, B, C, H, H, N, kind, depth, arity, K, pad,
                                                     pool, want_gx)


# (the plans follow the device's LDS: on a GPU) the paths within a few per cent of the shortest at these sizes
@pytest.mark.gpu
@pytest.mark.parametrize("paths,size", [
    ((SAMPLES,), (1024, 64, 14, 128, ops.GATE16, 2, 2, 4, 1, 1)),
    ((SAMPLES,), (512, 128, 16, 256, ops.MULTILINEAR2, 1, 6, 4, 1, 1)),
    ((SAMPLES,), (256, 64, 14, 128, ops.WALSH, 2, 2, 4, 1, 1)),
    ((SAMPLES,), (64, 2048, 8, 2048, ops.GATE16, 2, 2, 4, 1, 1)),
    ((SAMPLES,), (4096, 3, 32, 64, ops.GATE16, 2, 2, 4, 1, 1)),
    ((GENERIC,), (2, 448, 98, 11, ops.GATE16, 2, 2, 1, 0, 1)),            # 816 / 1316 / 83 us
    ((GENERIC,), (1, 77, 112, 116, ops.MULTILINEAR2, 1, 4, 4, 1, 0)),     # 2930 / - / 263
    ((POSITIONS,), (3, 4, 73, 395, ops.MULTILINEAR2, 1, 6, 5, 3, 1)),     # 8537 / 808 / 11902
    ((POSITIONS,), (5, 6, 53, 108, ops.MULTILINEAR2, 1, 5, 8, 2, 1)),     # 816 / 371 / 2905
    ((POSITIONS, GENERIC), (2, 82, 50, 358, ops.GATE16, 2, 2, 4, 2, 0)),  # 2004 / 439 / 310
    ((GENERIC,), (1, 323, 38, 170, ops.WALSH, 3, 2, 5, 2, 0)),            # 1141 / - / 179
])
def test_conv_backward_takes_the_shorter_kernels(paths, size):
    got = _floats(AUTO, *size)
    assert got in [_floats(p, *size) for p in paths]
    others = [_floats(p, *size) for p in (SAMPLES, POSITIONS, GENERIC) if p not in paths]
    assert got not in others


def test_a_call_without_input_gradient_reserves_none():
    size = (512, 3, 32, 64, ops.GATE16, 2, 2, 4, 1, 1)
    with_gx, without = _floats(AUTO, *size), _floats(AUTO, *size, 0)
    leaf_gradients = 512 * 64 * 4 * 16 * 16
    assert with_gx - without >= leaf_gradients
    assert with_gx == _lib.lib().slg_conv_soft_bwd_workspace(512, 3, 32, 32, *size[3:])


@pytest.mark.parametrize("size", [
    (65536, 512, 8, 8, ops.GATE16, 2, 2, 4, 1, 1),       # few trees under many channels
    (4096, 64, 32, 512, ops.MULTILINEAR2, 1, 6, 4, 1, 1),
])
def test_rounds_bound_the_workspace(size):
    # 96 M floats of a round, the partial sums of its jobs and the tables
    assert 0 < _floats(SAMPLES, *size) < 112 << 20


def test_refusals():
    size = (4, 3, 8, 4, ops.WALSH, 2, 2, 4, 1, 1)
    assert _floats(POSITIONS, *size) == -1 and _floats(4, *size) == -1 and _floats(-1, *size) == -1
    assert _floats(AUTO, 4, 3, 8, 4, ops.WALSH, 6, 2, 4, 1, 1) == -1
