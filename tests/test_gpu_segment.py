"""Segmentation on the device against the oracle, voxel for voxel: the
inverse-gradient region growing (with its closing) and the sphere
segmentation, on a synthetic tube field, a GVF field of rendered tubes, and
the 16-bit storage of that field."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tube_field(shape, peak):
    z, y, x = np.mgrid[:shape[0], :shape[1], :shape[2]].astype(np.float32)
    dy, dz = y - (shape[1] - 1) / 2, z - (shape[0] - 1) / 2
    rho = np.sqrt(dy * dy + dz * dz)
    m = np.where(rho <= peak, rho, np.maximum(0.0, 2 * peak - rho))
    F = np.zeros((4,) + shape, np.float32)
    with np.errstate(invalid="ignore", divide="ignore"):
        F[1] = np.where(rho > 0, -m * dy / rho, 0.0)
        F[2] = np.where(rho > 0, -m * dz / rho, 0.0)
    w = np.sqrt(F[1] ** 2 + F[2] ** 2)
    F[3] = np.where(w > 0, w, 1.0)
    return F


def run_device(tsf, cl, radius, F, storage=None):
    fld = tsf.Field.from_host(F) if storage is None else tsf.Field.from_host(F, storage[0], storage[1])
    out = tsf.DeviceArray(cl.shape, np.uint8)
    passes = tsf.segment_inverse_gradient(tsf.DeviceArray.from_host(cl), tsf.DeviceArray.from_host(radius), fld, out)
    return out.download(), passes


@pytest.mark.parametrize("nx", [32, 31], ids=["words", "bytes"])
def test_segment_tube_vs_oracle(tsf, orc, nx):
    """X = 32 takes the closing on 4-voxel words, X = 31 the byte passes."""
    shape = (28, 28, nx)
    F = tube_field(shape, 6.0)
    cl = np.zeros(shape, np.uint8)
    cl[13:15, 13:15, 2:30] = 1
    r = np.full(shape, 2.0, np.float32)
    got, passes = run_device(tsf, cl, r, F)
    exp, opasses = orc.segment_inverse_gradient(cl, r, F)
    print(f"tube: {int(got.sum())} voxels, {passes} passes (oracle {opasses})")
    assert passes == opasses and np.array_equal(got, exp)


@pytest.mark.parametrize("seed", [31, 32])
def test_segment_gvf_of_tubes_vs_oracle(tsf, orc, seed):
    # the GVF field of rendered tubes and a centerline from their skeleton
    from tsf import synth
    shape = (40, 44, 48)
    vol, _ = synth.tube_volume(shape, 5, 1.5, 3.5, seed, noise=0.02)
    F = orc.gvf_euler(orc.vector_field(orc.blur(vol, 0.5, "f32"), 0.2, 1, "f32"), 0.05, 40, "f32")
    t, rad = orc.tdf_circle(F, 1.0, 4.0, 0.5, "f32")
    cl = (t > np.quantile(t, 0.985)).astype(np.uint8)
    got, passes = run_device(tsf, cl, rad, F)
    exp, opasses = orc.segment_inverse_gradient(cl, rad, F)
    iou = (got & (vol > 0.5)).sum() / max((got | (vol > 0.5)).sum(), 1)
    print(f"tubes {seed}: {int(cl.sum())} centerline voxels -> {int(got.sum())} segmented, {passes} passes, "
          f"IoU with the tubes {iou:.3f}")
    assert passes == opasses and np.array_equal(got, exp)
    # the sphere segmentation of the same centerline
    s = tsf.DeviceArray(shape, np.uint8)
    tsf.segment_spheres(tsf.DeviceArray.from_host(cl), tsf.DeviceArray.from_host(rad), s)
    assert np.array_equal(s.download(), orc.segment_spheres(cl, rad))


def test_segment_reads_16bit_fields(tsf, orc):
    # an SN16 field: the device decodes the codes; the oracle gets the decoded values
    shape = (28, 28, 32)
    F = tube_field(shape, 6.0)
    F[:3] /= 8.0
    F[3] = np.where(np.sqrt((F[:3] ** 2).sum(0)) > 0, np.sqrt((F[:3] ** 2).sum(0)), 1.0)
    Fq = orc.sn16_round(F)
    cl = np.zeros(shape, np.uint8)
    cl[13:15, 13:15, 2:30] = 1
    r = np.full(shape, 2.0, np.float32)
    got, passes = run_device(tsf, cl, r, Fq, storage=(tsf.STORAGE_SN16, 1.0))
    exp, opasses = orc.segment_inverse_gradient(cl, r, Fq)
    assert passes == opasses and np.array_equal(got, exp)


@pytest.mark.parametrize("nx,half,step", [(8, 16, 1), (13, 16, 1), (4, 4, 1), (5, 1, 1), (68, 8, 2)],
                         ids=["two-batches", "odd-rows", "dense", "dense-odd", "sparse-seeds"])
def test_segment_lists_and_dense_passes(tsf, orc, nx, half, step):
    """Growing on lists over more than one batch of passes, and volumes whose
    candidates overflow the lists (seeds of half size 1..4 in a volume little
    larger than them), at row lengths with and without whole words."""
    side = 2 * half + 2
    shape = (side, side + 1, nx)
    F = tube_field(shape, 0.75 * half)
    cl = np.zeros(shape, np.uint8)
    cl[side // 2, side // 2, ::step] = 1
    r = np.full(shape, 2.0 if half > 4 else 2.0 * half, np.float32)
    got, passes = run_device(tsf, cl, r, F)
    exp, opasses = orc.segment_inverse_gradient(cl, r, F)
    print(f"{shape}: {int(got.sum())} voxels, {passes} passes (oracle {opasses})")
    assert passes == opasses and np.array_equal(got, exp)


@pytest.mark.parametrize("cells,side", [(1, 15), (1, 16), (4, 15), (4, 16)])
def test_segment_list_overflow_while_growing(tsf, orc, cells, side):
    """Seeds that fit the list (a quarter of the volume) and a first pass whose
    nominations do not: cells**3 basins, each seeded by a cube of 9**3 - 1
    around its centre, the field pointing there."""
    n = cells * side
    ax = (np.arange(n) % side - (side - 1) // 2).astype(np.float32)
    d = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"))[::-1]  # x, y, z
    rho = np.sqrt((d * d).sum(0))
    m = (np.where(rho <= 6, rho, np.maximum(0, 12 - rho)) / 32).astype(np.float32)
    F = np.zeros((4, n, n, n), np.float32)
    F[:3] = -m * d / np.where(rho > 0, rho, 1)
    F[3] = np.where(m > 0, m, 1e-3)
    cl = (rho == 0).astype(np.uint8)
    # the voxels that the first pass nominates: not the centre, pointing at a
    # seed of smaller magnitude
    cap = (n ** 3 + 255) // 256 * 64
    seeds = np.abs(d).max(0) <= 4
    dirs = np.array([(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1) if (a, b, c) != (0, 0, 0)])
    unit = dirs / np.sqrt((dirs ** 2).sum(1))[:, None]
    to = dirs[np.tensordot(unit, F[:3], 1).argmax(0)]  # (..., 3): x, y, z
    at = [np.clip(i + to[..., 2 - k], 0, n - 1) for k, i in enumerate(np.indices(F.shape[1:]))]
    nominated = (rho > 0) & seeds[tuple(at)] & (cl[tuple(at)] == 0) & (F[3] > F[3][tuple(at)])
    assert seeds.sum() - cl.sum() <= cap < nominated.sum()
    got, passes = run_device(tsf, cl, np.full(cl.shape, 8.0, np.float32), F)
    exp, opasses = orc.segment_inverse_gradient(cl, np.full(cl.shape, 8.0, np.float32), F)
    assert passes == opasses and np.array_equal(got, exp)


@pytest.mark.parametrize("seed", [5, 6])
def test_segment_direction_ties_vs_oracle(tsf, orc, seed):
    """Fields of small whole numbers: equal and zero components, zero vectors
    and vectors far from unit length, where the direction that a neighbour
    points at hangs on rounding and on the order of the 26."""
    g = np.random.default_rng(seed)
    shape = (24, 26, 28)
    F = np.zeros((4,) + shape, np.float32)
    F[:3] = g.integers(-2, 3, (3,) + shape)
    F[3] = g.choice([0.5, 1.0, 1.5, 3.0], shape)
    F[:3, :, :, 14:] *= np.float32(1e-33) if seed == 5 else np.float32(1.1)
    cl = (g.random(shape) < 0.01).astype(np.uint8)
    r = g.uniform(1.0, 5.0, shape).astype(np.float32)
    got, passes = run_device(tsf, cl, r, F)
    exp, opasses = orc.segment_inverse_gradient(cl, r, F)
    print(f"{int(cl.sum())} centerline voxels -> {int(got.sum())}, {passes} passes (oracle {opasses})")
    assert passes == opasses and np.array_equal(got, exp)
