"""GPU: the centerline stages at the sizes where their kernels change shape,
against the oracle, bit for bit."""
import numpy as np
import pytest
import scipy.ndimage as ndi

pytestmark = pytest.mark.gpu


def _dev(tsf, a):
    return tsf.DeviceArray.from_host(np.ascontiguousarray(a))


@pytest.mark.parametrize("cap", [1, 2, 3, 8, 20])
def test_nms_reach(tsf, orc, cap):
    # radii 0..24 on a smooth field: reaches of 1 (always kept), 2 (the 26
    # neighbours only) and wider (a wave per survivor), borders included
    shape = (26, 30, 33)
    g = np.random.default_rng(cap)
    V = np.stack([ndi.gaussian_filter(g.standard_normal(shape), 2.0) for _ in range(3)]).astype(np.float32)
    V = np.concatenate([V, np.linalg.norm(V, axis=0)[None].astype(np.float32)])
    V[3] = ndi.gaussian_filter(V[3], 3.0)  # minima of every reach
    tdf = g.uniform(0, 1, shape).astype(np.float32)
    rad = g.uniform(0, 24, shape).astype(np.float32)
    mask = (g.uniform(0, 1, shape) < 0.2).astype(np.uint8)
    mask[0, 0, 0] = mask[-1, -1, -1] = 1
    pos = orc.hp_compact(mask, "sort")
    out = tsf.DeviceArray(shape, np.uint8)
    out.zero()
    tsf.candidate_nms(_dev(tsf, tdf), _dev(tsf, rad), tsf.Field.from_host(V), _dev(tsf, pos), len(pos), cap, out)
    assert np.array_equal(out.download(), orc.candidate_nms(tdf, rad, V, pos, cap, "f32"))


@pytest.mark.parametrize("axis", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1), (1, -1, 0)])
def test_nms_straight_tubes(tsf, orc, axis):
    """Offsets in the plane across the tube and along its axis, where the
    cosine of their angle to the plane rounds to more than 1 (its arc cosine
    is NaN and the offset does not count) or is made of rounding errors.  A
    cell of 15^3 for each: a candidate in its middle and one darker voxel."""
    e = np.array(axis) / np.linalg.norm(axis)
    k = np.arange(-7, 8)
    r = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)  # x, y, z
    r2 = (r * r).sum(1)
    along = (r @ e) ** 2
    r = r[(r2 > 0) & (r2 < 64) & ((along <= 0.02 * r2) | (along >= 0.98 * r2))]
    m = int(np.ceil(len(r) ** (1 / 3)))
    n = 15 * m
    c = np.indices((n, n, n))[::-1] % 15 - 7.0  # x, y, z from the middle of the cell
    F = np.ones((4, n, n, n), np.float32)
    F[:3] = -(c - e[:, None, None, None] * np.tensordot(e, c, 1)) / 20
    cell = np.stack(np.unravel_index(np.arange(len(r)), (m, m, m)), 1)[:, ::-1]
    pos = np.ascontiguousarray(15 * cell + 7, np.int32)
    F[3][tuple((pos + r).T[::-1])] = 0.5
    rad = np.full((n, n, n), 8, np.float32)
    out = tsf.DeviceArray((n, n, n), np.uint8)
    out.zero()
    tsf.candidate_nms(_dev(tsf, rad), _dev(tsf, rad), tsf.Field.from_host(F), _dev(tsf, pos), len(pos), 8, out)
    exp = orc.candidate_nms(rad, rad, F, pos, 8, "f32")
    across = (r @ e) ** 2 < 1e-6
    kept = exp[tuple(pos.T[::-1])][across]
    assert 0 < kept.sum() < len(kept)
    assert np.array_equal(out.download(), exp)


@pytest.mark.parametrize("shape", [(9, 11, 516), (10, 7, 131), (5, 5, 8), (65, 66, 68)])
@pytest.mark.parametrize("cube", [1, 4, 5, 7, 64])
def test_cube_max_rows(tsf, orc, shape, cube):
    # rows of whole words and ragged ones, more columns than a workgroup, ties
    g = np.random.default_rng(cube)
    tdf = (g.integers(-1, 6, shape) / 4.0).astype(np.float32)
    cand = g.integers(0, 3, shape).astype(np.uint8)  # 2 is no candidate
    out = tsf.DeviceArray(shape, np.uint8)
    out.zero()
    tsf.cube_max(_dev(tsf, tdf), _dev(tsf, cand), cube, out)
    assert np.array_equal(out.download(), orc.cube_max(tdf, cand, cube, "f32"))


@pytest.mark.parametrize("n", [1, 3, 4, 4099])
def test_candidates_remainder(tsf, n):
    t = np.random.default_rng(n).uniform(0, 1, (1, 1, n)).astype(np.float32)
    t[0, 0, -1] = np.nan
    m = tsf.DeviceArray((1, 1, n), np.uint8)
    tsf.candidates(_dev(tsf, t), m, 0.5)
    assert np.array_equal(m.download(), np.where(t < 0.5, 0, 1))


@pytest.mark.parametrize("shape", [(3, 4, 300), (280, 6, 9), (2, 1030, 3)])
def test_compaction_of_many_cubes(tsf, orc, shape):
    # 32^3 cubes (eight tiles of the scan, a workgroup each), and 128^3 (one
    # workgroup for all tiles)
    m = (np.random.default_rng(1).uniform(0, 1, shape) < 0.3).astype(np.uint8)
    exp = orc.hp_compact(m, "sort")
    pos = tsf.DeviceArray((len(exp), 3), np.int32)
    assert tsf.hp_compact(_dev(tsf, m), pos) == len(exp)
    assert np.array_equal(pos.download(), exp)


def test_link_long_rows(tsf, orc):
    # hundreds of neighbours per vertex, several chunks of a wave
    g = np.random.default_rng(6)
    v = np.unique(g.integers(0, 14, (700, 3)).astype(np.int32), axis=0)
    T = ndi.gaussian_filter(g.standard_normal((14, 14, 14)), 1.0).astype(np.float32)
    T = (T - T.min()) / (T.max() - T.min())
    exp = orc.link_centerpoints(v, T, 12.0, 0.45)
    edges = tsf.DeviceArray((len(exp), 2), np.int32)
    assert tsf.link_centerpoints(_dev(tsf, v), len(v), _dev(tsf, T), 12.0, 0.45, edges) == len(exp)
    assert np.array_equal(edges.download(), exp)


@pytest.mark.parametrize("count", [16384, 16385])
def test_components_beyond_lds(tsf, orc, count):
    g = np.random.default_rng(count)
    e = np.stack([np.arange(1, count), np.arange(count - 1)], 1).astype(np.int32)
    e = e[g.uniform(0, 1, len(e)) < 0.97]
    labels, sizes = tsf.DeviceArray((count,), np.int32), tsf.DeviceArray((count,), np.int32)
    tsf.graph_components(_dev(tsf, e), len(e), count, labels, sizes)
    L, S = orc.graph_components(e, count)
    assert np.array_equal(labels.download(), L) and np.array_equal(sizes.download(), S)
