"""GPU: several GVF iterations per launch against single-step launches, bit for
bit, at extents around the multi-step kernel's tiles (64 columns, 8 to 24
rows) and on a volume large enough for its three-rows-per-thread form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32, SN16 = 0, 3


def _field(shape, seed):
    g = np.random.default_rng(seed)
    F = g.uniform(-0.7, 0.7, (4,) + shape).astype(np.float32)
    F[3] = 1.0
    return F


def _both(tsf, shape, iters, storage):
    f = tsf.Field.from_host(_field(shape, sum(shape)), storage)
    one, many = tsf.Field(shape, storage), tsf.Field(shape, storage)
    tsf.gvf_euler(f, one, 0.05, iters, fuse=1)
    tsf.gvf_euler(f, many, 0.05, iters, fuse=4)
    for a, b in zip(one.planes, many.planes):
        assert np.array_equal(a.download(), b.download())


@pytest.mark.parametrize("storage", [F32, SN16])
@pytest.mark.parametrize("shape,iters", [
    ((4, 4, 4), 5), ((5, 8, 63), 6), ((6, 9, 64), 7), ((7, 7, 65), 8), ((64, 16, 66), 9), ((13, 17, 67), 10),
    ((12, 23, 120), 11), ((66, 24, 121), 4), ((10, 25, 122), 3), ((30, 40, 128), 2), ((9, 41, 177), 13)])
def test_tile_edges(tsf, shape, iters, storage):
    _both(tsf, shape, iters, storage)


@pytest.mark.parametrize("shape,iters,storage", [((200, 401, 301), 7, F32), ((150, 300, 290), 5, SN16)])
def test_large_volume(tsf, shape, iters, storage):
    _both(tsf, shape, iters, storage)


@pytest.mark.parametrize("shape", [(20, 24, 66), (17, 30, 131)])
def test_every_state_of_a_segment(tsf, shape):
    # the adjoint recomputes a segment's iterates with launches that store all
    # of them: a segment of every iterate equals segments of one
    f = tsf.Field.from_host(_field(shape, 3)[:3])
    N = 9
    dV = tsf.DeviceArray.from_host(np.random.default_rng(4).standard_normal((3,) + shape).astype(np.float32))
    res = []
    for every in (N, 1):
        V = tsf.Field(shape)
        cps = tsf.DeviceArray((tsf.gvf_checkpoint_count(N, every), 3) + shape, np.float32)
        tsf.gvf_euler_checkpointed(f, V, 0.05, N, every, cps)
        dF = tsf.DeviceArray((3,) + shape, np.float32)
        dmu = tsf.gvf_euler_adjoint(f, 0.05, N, every, cps, dV, dF)
        res.append((V.download(), dF.download(), dmu))
    assert np.array_equal(res[0][0], res[1][0])
    assert np.array_equal(res[0][1], res[1][1])
    assert abs(res[0][2] - res[1][2]) <= 1e-9 * max(1.0, abs(res[1][2]))
