"""GPU parity of the affine transform and mask (through the C ABI): every
output sample bit-exact against the FP64-coordinate oracle, for both bit
depths, through the GPU-resident entry point and through transform_cuda_*'s
file output; the mask plane within one float ulp of the FP64 oracle."""
import os

import numpy as np
import pytest

from gpu_util import empty_device, from_device, to_device

pytestmark = pytest.mark.gpu

IDENT = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 1, 0]], np.float32)


def affine(seed, shape, rot=15.0):
    from gpu_deconvolution_amd.synth import random_affine
    return random_affine(np.random.default_rng(seed), shape, max_rot_deg=rot, max_shift=4.0)


def volume(shape, bits, seed):
    rng = np.random.default_rng(seed)
    maxv = (1 << bits) - 1
    v = rng.integers(0, maxv + 1, size=shape)
    v.reshape(-1)[:8] = [0, maxv, maxv - 1, 1 << (bits - 1), (1 << (bits - 1)) - 1, 1, 2, 3]
    return v.astype(np.uint16 if bits == 16 else np.uint8)


MATS = {
    "identity": lambda s: IDENT,
    "shift": lambda s: np.array([[1, 0, 0, 3], [0, 1, 0, -2], [0, 0, 1, 1]], np.float32),
    "halfvoxel": lambda s: np.array([[1, 0, 0, 0.5], [0, 1, 0, 0.5], [0, 0, 1, -0.5]], np.float32),
    "affine1": lambda s: affine(1, s),
    "affine2": lambda s: affine(2, s),
    "scale": lambda s: np.array([[1.1, 0, 0, -1.0], [0, 0.93, 0, 0.7], [0, 0, 1.05, 0.2]], np.float32),
}


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("name", list(MATS))
def test_transform_device_bit_exact(fm, orc, bits, name):
    shape = (24, 40, 56)
    tshape = (20, 44, 50)
    src = volume(shape, bits, seed=len(name) + bits)
    M = MATS[name](shape)
    print(f"\n[transform] bits={bits} mat={name}", flush=True)
    dt = np.uint16 if bits == 16 else np.uint8
    dsrc = to_device(src)
    ddst = empty_device(tshape, dt)
    fm.transform_device(dsrc.ptr, shape, ddst.ptr, tshape, M, bits=bits,
                        stream=0)
    fm.device_synchronize()
    got = from_device(ddst, dt)
    want = orc.transform(src.astype(np.uint16), M, tshape, bits=bits).astype(dt)
    assert np.array_equal(got, want), int(np.count_nonzero(got != want))


def test_transform_file_api_and_mask(fm, orc, tmp_path):
    shape = (30, 33, 47)
    tshape = (26, 35, 41)
    src = volume(shape, 16, seed=5)
    M = affine(7, shape)
    out = str(tmp_path / "out.raw")
    maskf = str(tmp_path / "mask.raw")
    fm.transform_to_file(src, M, tshape, out, mask_file=maskf, border=6, zspacing=2.5)
    got = np.fromfile(out, np.uint16).reshape(tshape)
    want = orc.transform(src, M, tshape)
    assert np.array_equal(got, want)
    mask = np.fromfile(maskf, np.float32).reshape(tshape[1:])
    mwant = orc.mask(shape, tshape, M, 6, 2.5)
    assert np.abs(mask - mwant).max() <= 2 * np.finfo(np.float32).eps
    assert (mask > 0).any() and (mask == 0).any()


def test_transform_file_api_8bit_many_chunks(fm, orc, tmp_path):
    # enough target planes that the driver writes several double-buffered chunks
    shape = (20, 300, 310)
    tshape = (2100, 256, 256)
    src = volume(shape, 8, seed=8)
    M = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0.01, 0]], np.float32)
    out = str(tmp_path / "o8.raw")
    fm.transform_to_file(src, M, tshape, out)
    got = np.fromfile(out, np.uint8).reshape(tshape)
    for z in (0, 1, 1023, 1024, 2099):
        want = orc.transform(src.astype(np.uint16), M, tshape, bits=8, z0=z, nz=1)[0].astype(np.uint8)
        assert np.array_equal(got[z], want), z


def test_mask_device(fm, orc):
    shape, tshape = (40, 50, 60), (30, 52, 64)
    M = affine(3, shape)
    d = empty_device(tshape[1:], np.float32)
    fm.mask_device(shape, tshape, M, 10, 1.5, d.ptr, stream=0)
    fm.device_synchronize()
    got = from_device(d, np.float32)
    assert np.abs(got - orc.mask(shape, tshape, M, 10, 1.5)).max() <= 2 * np.finfo(np.float32).eps


def test_transform_global_gather_fallback(fm, orc):
    """A map that magnifies by 2 and rotates by 45 deg about z makes every
    16 x 16 x 8 tile's source box exceed the largest LDS brick, so the kernel
    gathers from global memory; results stay bit-exact."""
    shape = (40, 120, 130)
    tshape = (18, 40, 44)
    src = volume(shape, 16, seed=12)
    c, s = np.cos(np.pi / 4), np.sin(np.pi / 4)
    M = np.array([[2 * c, -2 * s, 0.0, 60.0], [2 * s, 2 * c, 0.0, 10.0], [0.0, 0.0, 2.0, 1.5]], np.float32)
    dsrc = to_device(src)
    ddst = empty_device(tshape, np.uint16)
    fm.transform_device(dsrc.ptr, shape, ddst.ptr, tshape, M, bits=16, stream=0)
    fm.device_synchronize()
    got = from_device(ddst, np.uint16)
    want = orc.transform(src, M, tshape, bits=16)
    assert (want > 0).mean() > 0.5
    assert np.array_equal(got, want), int(np.count_nonzero(got != want))


def rotated(angles, scale, src, dst):
    """Inverse map about the volume centres: rotations about x, y, z (degrees), then a scale."""
    a = np.deg2rad(angles)
    (cx, cy, cz), (sx, sy, sz) = np.cos(a), np.sin(a)
    A = scale * (np.array([[cz, -sz, 0], [sz, cz, 0], [0, 0, 1]]) @ np.array([[cy, 0, sy], [0, 1, 0], [-sy, 0, cy]])
                 @ np.array([[1, 0, 0], [0, cx, -sx], [0, sx, cx]]))
    b = np.array(src[::-1]) / 2 - A @ (np.array(dst[::-1]) / 2)
    return np.concatenate([A, b[:, None]], 1).astype(np.float32)


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("shape,tshape,angles,scale", [
    ((1, 1, 1), (1, 1, 1), (0, 0, 0), 1.0),
    ((3, 5, 8), (17, 16, 33), (5, -9, 12), 0.9),       # boxes partly and wholly outside the volume
    ((41, 64, 64), (33, 48, 47), (15, 15, -15), 1.1),  # rows on 16-byte boundaries, boxes inside and across faces
    ((40, 63, 61), (33, 47, 49), (-15, 10, 15), 1.0),  # odd rows
    ((30, 50, 66), (30, 50, 66), (45, 45, 45), 1.0),   # a box near the limit of the LDS
    ((50, 70, 80), (20, 30, 33), (10, 20, 30), 2.4),   # beyond it: the general kernel
    ((20, 30, 48), (40, 60, 90), (0, 0, 45), 0.4),
])
def test_transform_box_edges(fm, orc, bits, shape, tshape, angles, scale):
    """The boxes a workgroup stages: at the volume's faces, outside it, at both row
    alignments, at and beyond the size limit."""
    src = volume(shape, bits, seed=shape[2] + bits) if shape != (1, 1, 1) else np.full(
        shape, 1 << (bits - 1), np.uint16 if bits == 16 else np.uint8)
    M = rotated(angles, scale, shape, tshape)
    dsrc, ddst = to_device(src), empty_device(tshape, src.dtype)
    fm.transform_device(dsrc.ptr, shape, ddst.ptr, tshape, M, bits=bits)
    fm.device_synchronize()
    want = orc.transform(src.astype(np.uint16), M, tshape, bits=bits).astype(src.dtype)
    assert np.array_equal(from_device(ddst, src.dtype), want)


def check_bit_exact(fm, orc, src, tshape, M, bits):
    dsrc, ddst = to_device(src), empty_device(tshape, src.dtype)
    fm.transform_device(dsrc.ptr, src.shape, ddst.ptr, tshape, np.asarray(M, np.float32), bits=bits)
    fm.device_synchronize()
    want = orc.transform(src.astype(np.uint16), np.asarray(M, np.float32), tshape, bits=bits).astype(src.dtype)
    got = from_device(ddst, src.dtype)
    assert np.array_equal(got, want), (int(np.count_nonzero(got != want)), np.argwhere(got != want)[:4])
    return want


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("tshape", [(1, 40, 50), (2, 17, 33), (5, 16, 16), (15, 20, 70), (17, 3, 40), (33, 1, 1), (40, 5, 2),
                                    (1, 1, 100), (1, 70, 1)])
def test_transform_thin_targets(fm, orc, bits, tshape):
    """Targets of fewer than 16 voxels along an axis: the staged box covers the voxels there are."""
    for shape in ((36, 48, 64), (35, 47, 61)):
        src = volume(shape, bits, seed=sum(tshape) + bits)
        for angles, scale in (((0, 0, 0), 1.0), ((20, -30, 40), 1.2), ((0, 90, 0), 1.0)):
            want = check_bit_exact(fm, orc, src, tshape, rotated(angles, scale, shape, tshape), bits)
            assert want.any()


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_transform_boxes_beside_the_volume(fm, orc, bits, axis):
    """Boxes that lie outside the volume, touch it, or hold its last texel only, on either side of an axis."""
    tshape = (33, 35, 37)
    for shape in ((20, 24, 32), (19, 23, 29)):
        src = volume(shape, bits, seed=axis + bits)
        n, t = shape[::-1][axis], tshape[::-1][axis]
        seen = []
        for shift in (-3e4, -t - 1.0, -t, -t + 0.5, -t + 1.0, -17.0, -16.5, -15.5, n - 17.0, n - 1.0, n - 0.25, n, n + 1.0, 3e4, 1e7):
            M = IDENT.copy()
            M[axis, 3] = shift
            seen.append(check_bit_exact(fm, orc, src, tshape, M, bits).any())
        assert any(seen) and not all(seen)


def dyadic_ties(src, tshape, frac, bits):
    """Target voxels whose unrounded value is exactly n + 1/2 under the shift frac (multiples of 1/64): integer sums."""
    f = [int(round(x * 64)) for x in frac]
    a = src.astype(np.int64)
    for axis, k in zip((2, 1, 0), f):
        p = np.pad(a, [(0, 1 if i == axis else 0) for i in range(3)])
        lo, hi = (np.take(p, np.arange(a.shape[axis]) + i, axis) for i in (0, 1))
        a = lo * (64 - k) + hi * k
    m = ((1 << bits) - 1) << 18  # the value is a 2^bits / m
    ties = (2 * (a << bits)) % m == 0
    return ties & ((2 * (a << bits)) // m % 2 == 1)


@pytest.mark.parametrize("bits, frac, shape, depth", [
    (8, (1 / 8, 3 / 8, 5 / 8), (24, 40, 64), 24), (8, (1 / 8, 3 / 8, 5 / 8), (23, 41, 61), 13),
    (8, (1 / 8, 1 / 8, 1 / 8), (17, 40, 64), 17), (8, (3 / 8, 7 / 8, 1 / 8), (21, 40, 35), 21),
    (16, (1 / 64, 1 / 64, 1 / 32), (75, 256, 256), 75), (16, (3 / 64, 5 / 64, 1 / 32), (70, 257, 255), 67)])
def test_transform_ties_take_the_definition(fm, orc, bits, frac, shape, depth):
    """Samples that lie exactly on a rounding boundary, which the box kernel's arithmetic cannot decide: dyadic shifts make them
    (about 0.2 % of 8-bit samples, 8 in a million of 16-bit ones), at every place in a column of 8 planes and in
    the last, shorter ones."""
    src = volume(shape, bits, seed=shape[2] + depth)
    tshape = (depth,) + shape[1:]
    ties = dyadic_ties(src, tshape, frac, bits)[:depth]
    assert ties.sum() >= (20 if bits == 8 else 5), ties.sum()
    if bits == 8:
        assert set(np.nonzero(ties)[0] % 8) == set(range(8))
    M = IDENT.copy()
    M[:, 3] = frac
    check_bit_exact(fm, orc, src, tshape, M, bits)


@pytest.mark.parametrize("angles, scale", [((0, 0, 0), 1.7), ((0, 0, 0), 1.75), ((0, 0, 0), 1.9), ((3, 3, 3), 1.7), ((0, 0, 45), 1.5),
                                           ((0, 0, 20), 1.65), ((0, 0, 25), 1.65)])
@pytest.mark.parametrize("bits", [16, 8])
def test_transform_large_boxes_of_odd_rows(fm, orc, bits, angles, scale):
    """Boxes on both sides of 160 / 3 KiB with rows off the 16-byte boundaries, along and across the source rows."""
    shape, tshape = (60, 65, 77), (33, 37, 41)
    src = volume(shape, bits, seed=int(10 * scale) + bits)
    want = check_bit_exact(fm, orc, src, tshape, rotated(angles, scale, shape, tshape), bits)
    assert (want > 0).mean() > 0.3
