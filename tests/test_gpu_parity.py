"""GPU parity: every C-ABI entry point against the CPU oracle on the same
seeded inputs.

Tolerances (stated per test):
  * integer / mask / index outputs: bit-exact;
  * FP32 field, eigenvalue and TDF outputs: per voxel |a - b| <= 1e-4 |b| + 1e-7
    (the stated FP32 bar), and the L2-relative error is reported;
  * reduced-precision storage forms: error against the FP64 oracle is
    measured and bounded, not parity.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-4, 1e-7


def close(a, b, rtol=RTOL, atol=ATOL):
    """(count of elements outside the tolerance, L2-relative difference);
    equal values (infinities included) and NaN on both sides agree, a NaN
    on one side does not."""
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    with np.errstate(invalid="ignore"):
        ok = (a == b) | (np.isnan(a) & np.isnan(b)) | (np.abs(a - b) <= rtol * np.abs(b) + atol)
        fin = np.isfinite(a) & np.isfinite(b)
        rel = float(np.linalg.norm((a - b)[fin]) / max(np.linalg.norm(b[fin]), 1e-30))
    return int((~ok).sum()), rel


def rng(s):
    return np.random.default_rng(s)


def phantom(shape, seed, noise=0.1, n=6):
    from tsf import synth
    vol, _ = synth.tube_volume(shape, n, 1.0, 3.5, seed, noise=noise)
    return vol


def dev(tsf, a, dtype=None):
    return tsf.DeviceArray.from_host(a, dtype)


# ------------------------------------------------------------------ prep
@pytest.mark.parametrize("shape", [(20, 23, 37), (3, 2, 1), (17, 9, 70)])
@pytest.mark.parametrize("sigma", [0.5, 1.0, 1.5, 2.0, 2.6])  # mask half-widths 1..5
def test_blur(tsf, orc, sigma, shape):
    v = rng(1).standard_normal(shape).astype(np.float32)
    a, b = dev(tsf, v), tsf.DeviceArray(v.shape, np.float32)
    tsf.blur_gaussian(a, b, sigma)
    got = b.download()
    exp = orc.blur(v, sigma, "f32")
    nbad, rel = close(got, exp, 1e-6, 1e-7)
    assert nbad == 0, rel
    assert np.array_equal(got, exp)  # same summation order, no contraction


@pytest.mark.parametrize("sigma,n", [(0.5, 9500), (2.6, 5500)])
def test_blur_wide_plane(tsf, orc, sigma, n):
    """Planes so large that a brick's planes span 2 GiB or more: the kernel
    addresses them with 64-bit pointers instead of buffer offsets.  One
    plane, so every z offset clamps to it; crops of the oracle's blur agree
    with the volume's away from the crop's cut edges (and on the volume's
    own edges, where both clamp)."""
    v = rng(7).standard_normal((1, n, n)).astype(np.float32)
    a, b = dev(tsf, v), tsf.DeviceArray(v.shape, np.float32)
    tsf.blur_gaussian(a, b, sigma)
    got = b.download()
    m = int(np.ceil(sigma / 0.5))
    for y, x in [(0, 0), (n // 2 - 17, n // 3 + 5), (n - 40, n - 40)]:
        crop = np.ascontiguousarray(v[:, y:y + 40, x:x + 40])
        exp = orc.blur(crop, sigma, "f32")
        ylo, xlo = (0 if y == 0 else m), (0 if x == 0 else m)
        yhi, xhi = (40 if y + 40 == n else 40 - m), (40 if x + 40 == n else 40 - m)
        assert np.array_equal(got[:, y + ylo:y + yhi, x + xlo:x + xhi], exp[:, ylo:yhi, xlo:xhi])


@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.uint16, np.int16, np.float32])
def test_to_float(tsf, orc, dtype):
    info = np.iinfo(dtype) if np.dtype(dtype).kind in "iu" else None
    lo, hi = (info.min, info.max) if info else (-50, 300)
    d = rng(2).integers(lo, hi, (8, 9, 10), endpoint=True).astype(dtype)
    a, b = dev(tsf, d), tsf.DeviceArray(d.shape, np.float32)
    tsf.to_float(a, b, 10.0, 75.0)
    assert np.array_equal(b.download(), orc.to_float(d.astype(np.float64), 10.0, 75.0, "f32"))


@pytest.mark.parametrize("sign,fmax", [(1, 0.2), (-1, 0.1)])
def test_vector_field(tsf, orc, sign, fmax):
    v = phantom((24, 28, 32), 3)
    a = dev(tsf, v)
    F = tsf.Field(v.shape)
    tsf.create_vector_field(a, F, fmax, sign)
    got = F.download()
    exp = orc.vector_field(v, fmax, sign, "f32")
    assert np.array_equal(got, exp)


# ------------------------------------------------------------------ GVF Euler
def _field_from(orc, vol, fmax=0.2, sigma=0.5):
    return orc.vector_field(orc.blur(vol, sigma, "f32"), fmax, 1, "f32")


@pytest.mark.parametrize("shape,iters", [((64, 64, 64), 250), ((20, 24, 36), 7), ((16, 17, 18), 1), ((8, 8, 8), 0),
                                         ((5, 13, 130), 3), ((4, 9, 66), 4), ((37, 23, 65), 5), ((70, 6, 4), 2)])
def test_gvf_euler_f32(tsf, orc, shape, iters):
    F = _field_from(orc, phantom(shape, 4))
    f = tsf.Field.from_host(F)
    out = tsf.Field(shape)
    tsf.gvf_euler(f, out, 0.1, iters)
    got = out.download()
    exp = orc.gvf_euler(F, 0.1, iters, "f32")
    nbad, rel = close(got, exp)
    print(f"gvf {shape} iters={iters}: L2 rel {rel:.3e}, exact {np.mean(got == exp):.4f}")
    assert nbad == 0, rel


@pytest.mark.parametrize("fuse", [2, 4])
@pytest.mark.parametrize("shape,iters", [((64, 64, 64), 250), ((20, 24, 36), 7), ((16, 17, 18), 2), ((8, 8, 8), 3),
                                         ((5, 13, 130), 4), ((4, 9, 66), 5), ((37, 23, 65), 6), ((70, 6, 4), 2),
                                         ((4, 4, 4), 4), ((5, 5, 5), 3), ((67, 7, 63), 8), ((130, 20, 125), 10),
                                         ((9, 31, 57), 12), ((6, 11, 5), 9)])
def test_gvf_euler_fused_two_steps(tsf, orc, shape, iters, fuse):
    # two or four steps per launch (fuse 2 / 4) compute the same float
    # operations in the same order as single-step launches: F32 results are
    # identical
    F = _field_from(orc, phantom(shape, 4))
    f = tsf.Field.from_host(F)
    a, b = tsf.Field(shape), tsf.Field(shape)
    tsf.gvf_euler(f, a, 0.1, iters, fuse=1)
    tsf.gvf_euler(f, b, 0.1, iters, fuse=fuse)
    ga, gb = a.download(), b.download()
    print(f"fused{fuse} {shape} iters={iters}: identical {np.mean(ga == gb):.6f}")
    assert np.array_equal(ga, gb)
    nbad, rel = close(gb, orc.gvf_euler(F, 0.1, iters, "f32"))
    assert nbad == 0, rel


@pytest.mark.parametrize("fuse", [2, 4])
@pytest.mark.parametrize("storage,bound", [(1, 2e-3), (2, 2e-2)])
def test_gvf_euler_fused_reduced_precision(tsf, orc, storage, bound, fuse):
    shape = (48, 48, 48)
    F = _field_from(orc, phantom(shape, 6))
    scale = 2.0 ** 14 if storage == 1 else 1.0
    f = tsf.Field.from_host(F, storage, scale)
    out = tsf.Field(shape, storage, scale)
    tsf.gvf_euler(f, out, 0.05, 100, fuse=fuse)
    got = out.download()
    ref = orc.gvf_euler(F.astype(np.float64), 0.05, 100, "f64")
    rel = np.linalg.norm(got[:3] - ref[:3]) / np.linalg.norm(ref[:3])
    print(f"fused{fuse} storage {storage}: L2 rel error vs FP64 {rel:.3e}")
    assert rel < bound
    # the magnitude plane is |v| of the stored components, itself stored:
    # one rounding of the storage type (2^-11 FP16, 2^-8 BF16) after the
    # float magnitude
    v = got[:3].astype(np.float64)
    w = np.sqrt((v ** 2).sum(0))
    assert np.allclose(got[3], np.where(w > 0, w, 1.0), rtol=1.01 * (2.0 ** -8 if storage == 2 else 2.0 ** -11), atol=0)


def test_gvf_euler_workspace_supplied(tsf, orc):
    shape = (16, 20, 24)
    F = _field_from(orc, phantom(shape, 5))
    f = tsf.Field.from_host(F)
    out = tsf.Field(shape)
    ws = tsf.DeviceArray((tsf.gvf_euler_workspace_size(shape, 0),), np.uint8)
    s = tsf.Stream()
    tsf.gvf_euler(f, out, 0.15, 12, workspace=ws, stream=s)
    s.synchronize()
    nbad, rel = close(out.download(), orc.gvf_euler(F, 0.15, 12, "f32"))
    assert nbad == 0, rel


@pytest.mark.parametrize("storage,bound", [(1, 2e-3), (2, 2e-2)])
def test_gvf_euler_reduced_precision(tsf, orc, storage, bound):
    # mu = 0.05: the explicit scheme is stable for 12 mu + |f|^2 <= 2; with
    # mu = 0.1 and |f| near 1 it amplifies the checkerboard mode (in every
    # precision, as the reference does), which a 16-bit store turns into inf.
    shape = (48, 48, 48)
    F = _field_from(orc, phantom(shape, 6))
    scale = 2.0 ** 14 if storage == 1 else 1.0
    f = tsf.Field.from_host(F, storage, scale)
    out = tsf.Field(shape, storage, scale)
    tsf.gvf_euler(f, out, 0.05, 100)
    got = out.download()
    ref = orc.gvf_euler(F.astype(np.float64), 0.05, 100, "f64")
    rel = np.linalg.norm(got[:3] - ref[:3]) / np.linalg.norm(ref[:3])
    print(f"storage {storage}: L2 rel error vs FP64 {rel:.3e}")
    assert rel < bound


# ------------------------------------------------------------------ 16-bit mode
# The reference's default 16-bit vectors (kernels_no_3d_write.cl:9-21): the
# field and every GVF iterate are SNORM16; float arithmetic between stores.
# Parity is bit-exact: the oracle runs the same float operations with the same
# rounding to codes.
SN16 = 3


@pytest.mark.parametrize("sign,fmax", [(1, 0.2), (-1, 0.1)])
def test_vector_field_sn16(tsf, orc, sign, fmax):
    v = phantom((24, 28, 32), 3)
    F = tsf.Field(v.shape, SN16)
    tsf.create_vector_field(dev(tsf, v), F, fmax, sign)
    assert np.array_equal(F.download(), orc.vector_field_sn16(v, fmax, sign))


@pytest.mark.parametrize("shape,iters,mu,fuse", [
    ((48, 48, 48), 100, 0.1, 1), ((48, 48, 48), 100, 0.1, 2), ((64, 64, 64), 250, 0.05, 2),
    ((20, 24, 36), 7, 0.05, 1), ((37, 23, 65), 6, 0.1, 2), ((5, 13, 130), 5, 0.1, 2), ((4, 4, 4), 3, 0.05, 2),
    ((70, 6, 4), 2, 0.1, 1), ((130, 20, 125), 10, 0.05, 2), ((16, 17, 18), 0, 0.05, 2),
    ((48, 48, 48), 100, 0.1, 4), ((37, 23, 65), 11, 0.1, 4), ((5, 5, 5), 8, 0.05, 4), ((130, 20, 125), 14, 0.05, 4)])
def test_gvf_euler_sn16(tsf, orc, shape, iters, mu, fuse):
    F = orc.vector_field_sn16(orc.blur(phantom(shape, 4), 0.5, "f32"), 0.2, 1)
    f = tsf.Field.from_host(F, SN16)
    out = tsf.Field(shape, SN16)
    tsf.gvf_euler(f, out, mu, iters, fuse=fuse)
    got = out.download()
    exp = orc.gvf_euler_sn16(F, mu, iters)
    print(f"sn16 gvf {shape} iters={iters} mu={mu} fuse={fuse}: identical {np.mean(got == exp):.6f}, "
          f"saturated {np.mean(np.abs(exp[:3]) == 1.0):.5f}")
    assert np.array_equal(got, exp)


def test_gvf_euler_sn16_error_vs_fp64(tsf, orc):
    # mu = 0.05 (stable): the 16-bit iterate's error against the FP64 oracle on
    # the same (already 16-bit) input field, reported and bounded
    shape = (48, 48, 48)
    F = orc.vector_field_sn16(orc.blur(phantom(shape, 6), 0.5, "f32"), 0.2, 1)
    f = tsf.Field.from_host(F, SN16)
    out = tsf.Field(shape, SN16)
    tsf.gvf_euler(f, out, 0.05, 100, fuse=2)
    got = out.download()
    ref = orc.gvf_euler(F.astype(np.float64), 0.05, 100, "f64")
    rel = np.linalg.norm(got[:3] - ref[:3]) / np.linalg.norm(ref[:3])
    print(f"sn16: L2 rel error vs FP64 {rel:.3e}")
    assert rel < 2e-3


def test_tdf_sn16_field_and_unorm16(tsf, orc):
    shape = (32, 32, 32)
    V = orc.gvf_euler_sn16(orc.vector_field_sn16(orc.blur(phantom(shape, 9), 0.5, "f32"), 0.2, 1), 0.05, 40)
    fld = tsf.Field.from_host(V, SN16)
    assert np.array_equal(fld.download(), V)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    tsf.tdf_circle(fld, 1.0, 5.0, 0.5, t, r)
    et, er = orc.tdf_circle(V, 1.0, 5.0, 0.5, "f32")
    nbad, rel = close(t.download(), et)
    print(f"SN16 TDF exact fraction {np.mean(t.download() == et):.6f}")
    assert nbad == 0, rel
    assert np.array_equal(r.download(), er)
    # UNORM16 rounding of the TDF buffer: bit-exact on the same values
    x = np.concatenate([t.download().ravel(), rng(30).uniform(-0.5, 1.5, 10000).astype(np.float32),
                        np.array([np.nan, np.inf, -np.inf, 0.5, 1.0, 0.0], np.float32)])
    d = dev(tsf, x)
    tsf.tdf_round_unorm16(d)
    assert np.array_equal(d.download(), orc.unorm16_round(x))


# ------------------------------------------------------------------ FMG
@pytest.mark.parametrize("shape,levels", [((32, 32, 32), 2), ((24, 20, 28), 2), ((16, 16, 16), 1)])
def test_gvf_fmg(tsf, orc, shape, levels):
    F = _field_from(orc, phantom(shape, 7), fmax=0.2)
    f = tsf.Field.from_host(F)
    out = tsf.Field(shape)
    norms = tsf.gvf_fmg(f, out, 0.15, 3, levels=levels, norms=True)
    got = out.download()
    exp = orc.gvf_fmg(F, 0.15, 3, 1, 2, 2, levels, "f32")
    nbad, rel = close(got, exp, 1e-4, 1e-6)
    print(f"fmg {shape}: L2 rel {rel:.3e}; residual norms {norms[:, -1]}")
    assert nbad == 0, rel
    assert np.all(norms[:, 1:] <= norms[:, :-1] * 1.0001)


@pytest.mark.parametrize("shape,levels,sweeps", [
    ((4, 5, 6), 0, (1, 2, 2)), ((9, 10, 11), 2, (1, 2, 2)), ((12, 17, 21), 1, (2, 0, 1)), ((8, 40, 33), 2, (0, 1, 1)),
    ((16, 16, 66), 2, (1, 1, 0)), ((30, 5, 24), 2, (1, 0, 0)), ((13, 12, 7), 1, (3, 1, 1))], ids=str)
def test_gvf_fmg_shapes_and_sweeps(tsf, orc, shape, levels, sweeps):
    """Rows whose last cell starts a quad, ends one or lies inside it, extents
    of 4 and 5 (each boundary mirrors the other's neighbour), and sweep counts
    of zero, after which every cell of a grid is read and not just the black
    ones.  The arithmetic and its order are the oracle's: equal bits."""
    F = _field_from(orc, phantom(shape, 9), fmax=0.2)
    f, out = tsf.Field.from_host(F), tsf.Field(shape)
    tsf.gvf_fmg(f, out, 0.15, 2, levels, *sweeps)
    exp = orc.gvf_fmg(F, 0.15, 2, *sweeps, levels, "f32")
    assert np.array_equal(out.download(), exp)


def test_gvf_fmg_small_workspace(tsf, orc):
    """A workspace of five grids per level (short of three components') runs
    the components one by one; one below a component's is refused."""
    shape, levels = (20, 22, 40), 2
    F = _field_from(orc, phantom(shape, 11), fmax=0.2)
    f, out = tsf.Field.from_host(F), tsf.Field(shape)
    n = 5 * 4 * (20 * 22 * 40 + 32 ** 3 + 16 ** 3) + 10000
    assert n < tsf.gvf_fmg_workspace_size(shape, levels)
    tsf.gvf_fmg(f, out, 0.15, 2, levels, workspace=tsf.DeviceArray((n,), np.uint8))
    assert np.array_equal(out.download(), orc.gvf_fmg(F, 0.15, 2, 1, 2, 2, levels, "f32"))
    with pytest.raises(tsf.TSFError):
        tsf.gvf_fmg(f, out, 0.15, 2, levels, workspace=tsf.DeviceArray((n // 2,), np.uint8))


@pytest.mark.parametrize("shape,levels", [((20, 18, 4), 0), ((11, 40, 9), 0), ((5, 5, 5), 1), ((10, 6, 4), 1),
                                          ((4, 4, 4), 0), ((16, 16, 16), 2)])
def test_gvf_fmg_workspace_of_five_grids(tsf, orc, shape, levels):
    # five plain arrays of every level hold one component's padded ones but
    # for rows of 4 or 9 elements and the smallest volumes; a byte less than
    # both is refused
    F = _field_from(orc, phantom(shape, 11), fmax=0.2)
    five, one, dims = 8192 + 256, 8192 + 256, shape
    for _ in range(levels + 1):
        five += 5 * ((4 * int(np.prod(dims)) + 255) // 256 * 256)
        xs = ((dims[2] + 1) // 2 + 3) // 4 * 4
        one += 3 * ((8 * xs * dims[0] * dims[1] + 255) // 256 * 256)
        dims = ((1 << (max(dims) - 1).bit_length()) // 2,) * 3
    out = tsf.Field(shape)
    ws = tsf.DeviceArray.from_host(np.full(five + 4096, 0xa5, np.uint8))
    ws.nbytes = five
    tsf.gvf_fmg(tsf.Field.from_host(F), out, 0.15, 2, levels, workspace=ws)
    assert np.array_equal(out.download(), orc.gvf_fmg(F, 0.15, 2, 1, 2, 2, levels, "f32"))
    ws.nbytes = five + 4096
    assert np.all(ws.download()[five:] == 0xa5)
    ws.nbytes = min(five, one) - 1
    with pytest.raises(tsf.TSFError):
        tsf.gvf_fmg(tsf.Field.from_host(F), out, 0.15, 2, levels, workspace=ws)


def test_gvf_fmg_one_component_at_a_time(tsf):
    """Above 2^27 cells the components share one set of buffers: what one
    leaves there must not reach the next, so permuted components (with a zero
    one, which keeps the rounding of |F|^2) give permuted results."""
    shape = (513, 512, 512)
    g = np.random.default_rng(12)
    a, b = (np.resize(g.uniform(-0.2, 0.2, (9, 64, 512)).astype(np.float32), shape) for _ in range(2))
    o = np.zeros(shape, np.float32)
    got = []
    for comps in ((a, b, o), (b, o, a)):
        f, out = tsf.Field(shape), tsf.Field(shape)
        for d, c in zip(f.planes, comps):
            d.upload(c)
        tsf.gvf_fmg(f, out, 0.15, 1, 1)
        got.append([p.download() for p in out.planes[:3]])
    assert np.array_equal(got[0][0], got[1][2]) and np.array_equal(got[0][1], got[1][0])
    assert not got[0][2].any() and not got[1][1].any()


# ------------------------------------------------------------------ eigen / TDF
def _gvf_field(orc, shape, seed, iters=40, mu=0.1):
    F = _field_from(orc, phantom(shape, seed))
    return orc.gvf_euler(F, mu, iters, "f32")


@pytest.mark.parametrize("normalize", [0, 1])
def test_hessian_eigen(tsf, orc, normalize):
    shape = (20, 22, 24)
    V = _gvf_field(orc, shape, 8)
    fld = tsf.Field.from_host(V)
    lam = tsf.DeviceArray((3,) + shape, np.float32)
    vec = tsf.DeviceArray((9,) + shape, np.float32)
    tsf.hessian_eigen(fld, normalize, lam, vec)
    gl, gv = lam.download(), vec.download()
    el, ev = orc.hessian_eigen(V, normalize, prec="f32")
    print(f"eigen exact fraction: {np.mean(gl == el):.5f}")
    nbad, rel = close(gl, el)
    assert nbad == 0, rel
    nbad, rel = close(gv, ev, 1e-4, 1e-6)
    assert nbad == 0, rel


# rmax 6: halo 7, past the FP32 planes tile (texels gathered from device memory)
@pytest.mark.parametrize("rmin,rmax,rstep", [(1.0, 3.0, 0.5), (2.5, 5.0, 0.5), (0.5, 4.0, 1.0), (3.0, 6.0, 0.5)])
def test_tdf_circle(tsf, orc, rmin, rmax, rstep):
    shape = (32, 32, 32)
    V = _gvf_field(orc, shape, 9)
    fld = tsf.Field.from_host(V)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    tsf.tdf_circle(fld, rmin, rmax, rstep, t, r)
    gt, gr = t.download(), r.download()
    et, er = orc.tdf_circle(V, rmin, rmax, rstep, "f32")
    nbad, rel = close(gt, et)
    print(f"tdf exact fraction {np.mean(gt == et):.5f}, radius agree {np.mean(gr == er):.5f}, rel {rel:.2e}")
    assert nbad == 0, rel
    assert np.array_equal(gr, er)


@pytest.mark.parametrize("storage", [0, 1])  # F32 planes, F16 texels
@pytest.mark.parametrize("rmin,rmax", [(0.5, 3.0), (2.5, 4.0)])  # halos 4 and 5
@pytest.mark.parametrize("shape", [(23, 29, 37), (9, 5, 70)])
def test_tdf_circle_ragged(tsf, orc, shape, rmin, rmax, storage):
    """The reference-order TDF on volumes that are no multiple of its bricks
    (16 x 8 x 4; 16 x 16 x 4 for F32 planes at halo 5) and thinner than the
    halo in y: the partial bricks and the clamped tile against the oracle on
    the field's stored values."""
    V = _gvf_field(orc, shape, 13)
    fld = tsf.Field.from_host(V, storage, _f16_scale(V)) if storage else tsf.Field.from_host(V)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    tsf.tdf_circle(fld, rmin, rmax, 0.5, t, r)
    et, er = orc.tdf_circle(fld.download(), rmin, rmax, 0.5, "f32")
    assert np.isfinite(et).all()
    nbad, rel = close(t.download(), et)
    assert nbad == 0, rel
    assert np.array_equal(r.download(), er)


@pytest.mark.parametrize("mode", ["f32", "f16", "mixed"])
def test_tdf_wide_halo(tsf, orc, mode):
    """Radii 2.5-9 (halo 10): tiles too large for a workgroup's LDS, so the
    samples gather texels from device memory, against the oracle."""
    shape = (30, 34, 40)
    V = _gvf_field(orc, shape, 15)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    if mode == "mixed":
        fld = tsf.Field.from_host(V)
        scale = _f16_scale(V[:3])
        tsf.tdf_circle_mixed(fld, 2.5, 9.0, 0.5, t, r, sample_storage=1, sample_scale=scale)
        Vs = V.copy()
        Vs[:3] = orc.f16_round(V[:3], scale)
        et, er = orc.tdf_circle_mixed(V, Vs, 2.5, 9.0, 0.5, "f32")
        assert np.array_equal(t.download(), et) and np.array_equal(r.download(), er)
        return
    fld = tsf.Field.from_host(V, 1, _f16_scale(V)) if mode == "f16" else tsf.Field.from_host(V)
    tsf.tdf_circle(fld, 2.5, 9.0, 0.5, t, r)
    et, er = orc.tdf_circle(fld.download(), 2.5, 9.0, 0.5, "f32")
    assert np.isfinite(et).all() and (et > 0).sum() > 100
    nbad, rel = close(t.download(), et)
    assert nbad == 0, rel
    assert np.array_equal(r.download(), er)


@pytest.mark.parametrize("storage", [0, 1, 2, 3])
def test_tdf_gather_inside_and_at_the_faces(tsf, orc, storage):
    """Gathered samples in bricks that radius after radius lose their room
    inside the volume (unclamped taps, then clamped ones), every storage."""
    shape = (44, 50, 90)
    V = _gvf_field(orc, shape, 16)
    fld = tsf.Field.from_host(V, storage, 1.0 if storage in (0, 3) else _f16_scale(V))
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    tsf.tdf_circle(fld, 2.5, 18.0, 0.5, t, r)
    et, er = orc.tdf_circle(fld.download(), 2.5, 18.0, 0.5, "f32")
    assert np.isfinite(et).all() and (et > 0).sum() > 100
    assert np.array_equal(t.download(), et) and np.array_equal(r.download(), er)


def test_tdf_gather_wide_planes(tsf, orc):
    """Planes of more than 2^24 texels gather through 64-bit addresses: the
    corner of such a volume equals the same corner in a small one."""
    small, big = (3, 96, 96), (3, 4097, 4096)
    z, y, x = np.mgrid[:small[0], :small[1], :small[2]].astype(np.float32)
    V = np.full((4,) + small, 0.01, np.float32)  # a tube along z; 0.01 everywhere past row and column 80
    g = np.where((x < 80) & (y < 80), np.exp(-((x - 33) ** 2 + (y - 30) ** 2) / 50.0), 0.0) * (1 + 0.1 * z)
    V[0] += (33 - x) * g / 8
    V[1] += (30 - y) * g / 8
    V[3] = np.sqrt((V[:3] ** 2).sum(0))
    W = np.full((4,) + big, V[0, 0, 95, 95], np.float32)
    W[3] = V[3, 0, 95, 95]
    W[:, :, :96, :96] = V
    got = []
    for shape, F in ((small, V), (big, W)):
        t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
        tsf.tdf_circle(tsf.Field.from_host(F, 1, _f16_scale(V)), 2.5, 9.0, 0.5, t, r)
        got.append((t.download()[:, :70, :70], r.download()[:, :70, :70]))
    assert (got[0][0] > 0).sum() > 100
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("mode", ["f32", "f16", "mixed"])
def test_tdf_deep_volume(tsf, orc, mode):
    """A volume 5600 planes deep, where the compile-time-stride kernels'
    float cell addresses would pass 2^24 bytes: the launchers take the
    run-time-stride kernels, and the results still match the oracle."""
    shape = (5600, 6, 12)
    V = _gvf_field(orc, shape, 14, iters=10)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    if mode == "mixed":
        fld = tsf.Field.from_host(V)
        scale = _f16_scale(V[:3])
        tsf.tdf_circle_mixed(fld, 0.5, 3.0, 0.5, t, r, sample_storage=1, sample_scale=scale)
        Vs = V.copy()
        Vs[:3] = orc.f16_round(V[:3], scale)
        et, er = orc.tdf_circle_mixed(V, Vs, 0.5, 3.0, 0.5, "f32")
        assert np.array_equal(t.download(), et) and np.array_equal(r.download(), er)
        return
    fld = tsf.Field.from_host(V, 1, _f16_scale(V)) if mode == "f16" else tsf.Field.from_host(V)
    tsf.tdf_circle(fld, 0.5, 3.0, 0.5, t, r)
    et, er = orc.tdf_circle(fld.download(), 0.5, 3.0, 0.5, "f32")
    assert np.isfinite(et).all()
    nbad, rel = close(t.download(), et)
    assert nbad == 0, rel
    assert np.array_equal(r.download(), er)


def _f16_scale(V):
    """The power of two that keeps every value of V * scale inside F16's
    range (2^14 for fields within +-2)."""
    return float(2.0 ** min(14, np.floor(np.log2(32768.0 / max(float(np.abs(V).max()), 1e-30)))))


def _bf16_round(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


@pytest.mark.parametrize("storage,rmin,rmax", [(1, 1.0, 3.0), (1, 2.5, 4.0), (2, 0.5, 3.0), (2, 2.5, 5.0), (1, 3.0, 6.0)])
def test_tdf_circle_mixed(tsf, orc, storage, rmin, rmax):
    """Mixed mode: Hessian from the F32 field, samples from its 16-bit
    rounding with fused multiply-adds -- the oracle's mixed filter on the
    same two fields."""
    shape = (32, 32, 32)
    V = _gvf_field(orc, shape, 11)
    fld = tsf.Field.from_host(V)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    tsf.tdf_circle_mixed(fld, rmin, rmax, 0.5, t, r, sample_storage=storage,
                         sample_scale=2.0 ** 14 if storage == 1 else 1.0)
    gt, gr = t.download(), r.download()
    Vs = V.copy()
    Vs[:3] = orc.f16_round(V[:3]) if storage == 1 else _bf16_round(V[:3])
    et, er = orc.tdf_circle_mixed(V, Vs, rmin, rmax, 0.5, "f32")
    nbad, rel = close(gt, et)
    print(f"mixed TDF: exact fraction {np.mean(gt == et):.6f}, radius agree {np.mean(gr == er):.6f}")
    assert nbad == 0, rel
    assert np.array_equal(gr, er)


@pytest.mark.parametrize("storage", [1, 2])
@pytest.mark.parametrize("rmin,rmax", [(0.5, 3.0), (2.5, 4.0)])  # halos 4 and 5 (compile-time strides)
@pytest.mark.parametrize("shape", [(23, 29, 37), (9, 5, 70)])
def test_tdf_circle_mixed_ragged(tsf, orc, shape, rmin, rmax, storage):
    """Mixed mode on volumes that are no multiple of the bricks (16 x 8 x 4
    at halo 4, 8 x 8 x 8 at halo 5) and thinner than the halo in y: the
    partial bricks and the clamped tile against the oracle, F16 and BF16
    samples."""
    V = _gvf_field(orc, shape, 12)
    fld = tsf.Field.from_host(V)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    scale = _f16_scale(V[:3])
    tsf.tdf_circle_mixed(fld, rmin, rmax, 0.5, t, r, sample_storage=storage,
                         sample_scale=scale if storage == 1 else 1.0)
    gt, gr = t.download(), r.download()
    Vs = V.copy()
    Vs[:3] = orc.f16_round(V[:3], scale) if storage == 1 else _bf16_round(V[:3])
    et, er = orc.tdf_circle_mixed(V, Vs, rmin, rmax, 0.5, "f32")
    assert np.isfinite(et).all()
    assert np.array_equal(gt, et) and np.array_equal(gr, er)


@pytest.mark.parametrize("rmin,rmax", [(1.0, 3.0), (3.0, 6.0)])  # halos 4 and 7
@pytest.mark.parametrize("storage", [1, 2])
def test_tdf_reduced_precision_field(tsf, orc, storage, rmin, rmax):
    shape = (32, 32, 32)
    V = _gvf_field(orc, shape, 10)
    scale = 2.0 ** 14 if storage == 1 else 1.0
    fld = tsf.Field.from_host(V, storage, scale)
    t, r = tsf.DeviceArray(shape, np.float32), tsf.DeviceArray(shape, np.float32)
    tsf.tdf_circle(fld, rmin, rmax, 0.5, t, r)
    gt, gr = t.download(), r.download()
    # kernel parity given the same (quantised) field: FP32 oracle on fld's
    # values (exactly representable in float)
    Vq = fld.download()
    qt, qr = orc.tdf_circle(Vq, rmin, rmax, 0.5, "f32")
    nbad, rel = close(gt, qt)
    print(f"TDF on the stored field: exact fraction {np.mean(gt == qt):.6f}")
    assert nbad == 0, rel
    assert np.array_equal(gr, qr)
    # quantisation effect (reported): the first-maximum radius search is
    # discontinuous, so a few voxels change radius and dominate the L2 error
    et, er = orc.tdf_circle(V.astype(np.float64), rmin, rmax, 0.5, "f64")
    same = gr == er
    rel_all = np.linalg.norm(gt - et) / np.linalg.norm(et)
    rel_same = np.linalg.norm((gt - et)[same]) / np.linalg.norm(et[same])
    print(f"TDF storage {storage}: L2 rel vs FP64 {rel_all:.3e} (all), {rel_same:.3e} "
          f"(voxels whose radius did not change); radius changed at {int((~same).sum())} voxels")
    # radii from 4 up take the normalised Hessian, whose division by |v|
    # amplifies the storage rounding (oracle, radii 3-6: 2.2e-3 F16, 1.8e-2 BF16)
    assert rel_same < (2e-3 if storage == 1 else 2e-2) * (1 if rmax < 4 else 2)


def test_combine_candidates(tsf, orc):
    g = rng(11)
    shape = (10, 12, 14)
    ts, rs, tl, rl = (g.uniform(0, 1, shape).astype(np.float32) for _ in range(4))
    d = [dev(tsf, a) for a in (ts, rs, tl, rl)]
    tsf.combine(*d)
    et, er = orc.combine(ts, rs, tl, rl, "f32")
    assert np.array_equal(d[2].download(), et) and np.array_equal(d[3].download(), er)
    m = tsf.DeviceArray(shape, np.uint8)
    tsf.candidates(d[0], m, 0.5)
    assert np.array_equal(m.download(), orc.candidates(ts, 0.5, "f32"))


# ------------------------------------------------------------------ compaction
@pytest.mark.parametrize("shape,p", [((64, 64, 64), 0.05), ((20, 12, 28), 0.3), ((5, 9, 7), 0.5), ((100, 100, 100), 0.01),
                                     ((17, 33, 65), 1.0), ((16, 16, 16), 0.0), ((40, 24, 200), 0.002),
                                     ((48, 80, 32), 0.1), ((3, 2, 4112), 0.3), ((2, 3, 4200), 0.3)])
def test_hp_compact_bit_exact(tsf, orc, shape, p):
    mask = (rng(12).uniform(0, 1, shape) < p).astype(np.uint8)
    n = int(mask.sum())
    m = dev(tsf, mask)
    pos = tsf.DeviceArray((max(n, 1), 3), np.int32)
    cnt = tsf.hp_compact(m, pos)
    assert cnt == n
    got = pos.download()[:n]
    exp = orc.hp_compact(mask, "sort")
    assert np.array_equal(got, exp)


def test_hp_compact_capacity(tsf, orc):
    mask = (rng(13).uniform(0, 1, (16, 16, 16)) < 0.2).astype(np.uint8)
    n = int(mask.sum())
    m = dev(tsf, mask)
    pos = tsf.DeviceArray((10, 3), np.int32)
    with pytest.raises(tsf.TSFError) as e:
        tsf.hp_compact(m, pos)
    assert e.value.status == 5
    assert np.array_equal(pos.download(), orc.hp_compact(mask, "sort")[:10])
    assert tsf.hp_compact(m, None) == n


def test_candidate_nms_and_cube_max(tsf, orc):
    shape = (32, 32, 32)
    V = _gvf_field(orc, shape, 14)
    et, er = orc.tdf_circle(V, 1.0, 3.0, 0.5, "f32")
    mask = orc.candidates(et, float(np.quantile(et, 0.9)), "f32")
    pos = orc.hp_compact(mask, "sort")
    fld = tsf.Field.from_host(V)
    t, r = dev(tsf, et), dev(tsf, er)
    p = dev(tsf, pos)
    for cap in (5, 8):
        out = tsf.DeviceArray(shape, np.uint8)
        out.zero()
        tsf.candidate_nms(t, r, fld, p, pos.shape[0], cap, out)
        got = out.download()
        exp = orc.candidate_nms(et, er, V, pos, cap, "f32")
        assert np.sum(got != exp) == 0
    cand = dev(tsf, exp)
    for cube in (3, 4, 5):
        o = tsf.DeviceArray(shape, np.uint8)
        o.zero()
        tsf.cube_max(t, cand, cube, o)
        assert np.array_equal(o.download(), orc.cube_max(et, exp, cube, "f32"))


def test_do_eigen_points(tsf, orc):
    shape = (12, 14, 16)
    V = _gvf_field(orc, shape, 15)
    pts = np.array([[3, 4, 5], [1, 1, 1], [14, 12, 10], [7, 7, 7]], np.int32)
    d = [dev(tsf, V[k]) for k in range(3)]
    out = tsf.DeviceArray((pts.shape[0], 12), np.float32)
    tsf.do_eigen_points(*d, dev(tsf, pts), out)
    got = out.download()
    for i, p in enumerate(pts):
        l, e1, e2, e3 = orc.do_eigen(V[0], V[1], V[2], p, "f32")
        exp = np.concatenate([l, e1, e2, e3])
        nbad, rel = close(got[i], exp, 1e-4, 1e-6)
        assert nbad == 0, (p, rel)
