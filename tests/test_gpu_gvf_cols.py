"""GPU: several GVF iterations per launch against single-step launches, bit for
bit, at extents around the multi-step kernel's tiles (64 columns, 8 to 24
rows) and on a volume large enough for its three-rows-per-thread form.  F16
and BF16 planes, which round other iterates, against the same on the host."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32, F16, BF16, SN16 = 0, 1, 2, 3


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


@pytest.mark.parametrize("shape,iters,storage", [
    ((200, 401, 301), 7, F32), ((150, 300, 290), 5, SN16),
    # few planes, narrow rows, both: within the last-level cache
    ((11, 310, 290), 9, F32), ((260, 250, 16), 7, F32), ((30, 1300, 31), 6, F32)])
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


def _step(v, f, mu):
    """One iteration in float32, in the kernels' order; every voxel takes the
    update of its mirror."""
    n = [slice(1, -1)] * 3
    s = np.float32(-6) * v[:, 1:-1, 1:-1, 1:-1]
    for axis in (3, 2, 1):
        for at in (slice(2, None), slice(None, -2)):
            k = [slice(None)] + n
            k[axis] = at
            s = s + v[tuple(k)]
    vi, fi = v[:, 1:-1, 1:-1, 1:-1], f[:, 1:-1, 1:-1, 1:-1]
    m2 = fi[0] * fi[0] + fi[1] * fi[1] + fi[2] * fi[2]
    new = vi + (np.float32(mu) * s - (vi - fi) * m2)
    m = [np.clip(np.where(np.arange(k) == 0, 2, np.where(np.arange(k) == k - 1, k - 3, np.arange(k))), 0, k - 1) - 1
         for k in v.shape[1:]]
    return new[np.ix_(range(3), *m)]


@pytest.mark.parametrize("storage,scale", [(F16, 2.0 ** 14), (BF16, 1.0)])
@pytest.mark.parametrize("shape,iters,fuse", [
    ((4, 4, 4), 11, 4), ((7, 7, 65), 11, 4), ((13, 17, 67), 7, 4), ((30, 24, 121), 6, 4), ((9, 41, 177), 8, 4),
    ((5, 8, 64), 5, 2), ((7, 9, 65), 4, 2), ((64, 16, 67), 3, 2), ((20, 33, 130), 6, 2), ((120, 180, 200), 2, 2)])
def test_16bit_tiles(tsf, shape, iters, fuse, storage, scale):
    """F16 and BF16 planes, whose iterates are rounded once per launch (the last
    shape takes two rows per thread): bit for
    bit the same in float32 on the host, rounded after a first single step, a
    pair and then every four iterations (fuse 4) or every two."""
    def rounded(v):
        w = np.ones((1,) + shape, np.float32)
        return tsf.Field.from_host(np.concatenate([v, w]), storage, scale).download()[:3]

    F = _field(shape, sum(shape) + iters)
    out = tsf.Field(shape, storage, scale)
    tsf.gvf_euler(tsf.Field.from_host(F, storage, scale), out, 0.05, iters, fuse=fuse)
    f = rounded(F[:3])
    fours = iters // 4 if fuse == 4 else 0
    rest = iters - 4 * fours
    v = f
    for k in [1] * (rest % 2) + [2] * (rest // 2) + [4] * fours:
        for _ in range(k):
            v = _step(v, f, 0.05)
        v = rounded(v)
    got = out.download()
    assert np.array_equal(got[:3], v)
    w = np.sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
    w = tsf.Field.from_host(np.concatenate([v, np.where(w > 0, w, 1)[None]]), storage, scale).download()[3]
    assert np.array_equal(got[3], w)
