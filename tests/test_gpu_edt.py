"""GPU EDT field (maxibone_amd/csrc/mxb_edt.hip) vs the oracle
(oracle/edt.py): exact squared distances, their float32 square roots and the
0950 uint16 field, bit for bit, through the C ABI, the Python drop-in and the
device entries."""
import sys

import numpy as np
import pytest

from maxibone_amd import capi, edt, hip
from maxibone_amd.helpers import generate_cylinder_mask
from oracle import edt as E

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


SHAPES = [(6, 7, 9), (1, 1, 13), (5, 1, 8), (9, 8, 1), (17, 33, 65), (64, 64, 64), (3, 130, 70),
          (40, 20, 129), (2, 300, 5), (70, 3, 257)]


@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_edt_sq_matches_oracle(gpu, case):
    rng = np.random.default_rng(900 + case)
    shape = SHAPES[case]
    density = [0.05, 0.2, 0.1, 0.3, 0.01, 0.002, 0.05, 0.02, 0.5, 0.001][case]
    data = rng.random(shape) > density
    data.flat[rng.integers(data.size)] = False
    _say("edt_sq", shape, density)
    want = E.edt_sq(data)
    got = edt.edt_sq(data)
    assert np.array_equal(got.astype(np.uint64), want)
    f = edt.edt(data)
    assert np.array_equal(f, E.edt(data))


@pytest.mark.parametrize("n", [1024, 2048, 4096])
def test_edt_long_axes(gpu, n):
    """Lines of 1024, 2048 and 4096 voxels (bands of 16, 32 and 64 per lane)
    along each axis in turn."""
    rng = np.random.default_rng(n)
    for axis in range(3):
        shape = [3, 4, 5]
        shape[axis] = n
        data = rng.random(shape) > 0.003
        data.flat[rng.integers(data.size)] = False
        _say("edt long axis", shape)
        assert np.array_equal(edt.edt_sq(data).astype(np.uint64), E.edt_sq(data))


def test_edt_no_site_and_all_sites(gpu):
    assert np.all(edt.edt_sq(np.ones((5, 6, 7), bool)) == edt.EDT_NONE)
    assert np.all(np.isinf(edt.edt(np.ones((5, 6, 7), bool))))
    assert np.all(edt.edt_sq(np.zeros((5, 6, 7), bool)) == 0)
    one = np.ones((9, 10, 11), bool)
    one[0, 0, 0] = False
    z, y, x = np.indices(one.shape)
    assert np.array_equal(edt.edt_sq(one), (z * z + y * y + x * x).astype(np.uint32))


def test_edt_ties_and_structured_sites(gpu):
    """Periodic and planar sites: many equal distances (ties in every pass)."""
    data = np.ones((24, 40, 56), bool)
    data[::7, ::5, ::3] = False
    assert np.array_equal(edt.edt_sq(data).astype(np.uint64), E.edt_sq(data))
    data = np.ones((24, 40, 56), bool)
    data[:, 13, :] = False
    data[5, :, 40] = False
    assert np.array_equal(edt.edt_sq(data).astype(np.uint64), E.edt_sq(data))


def _rod_implant(shape, rng):
    nz, ny, nx = shape
    implant = np.zeros(shape, bool)
    cy, cx, r = ny // 2, nx // 2, max(2, min(ny, nx) // 10)
    yy, xx = np.mgrid[:ny, :nx]
    implant[nz // 4:, (yy - cy) ** 2 + (xx - cx) ** 2 <= r * r] = True
    implant[rng.random(shape) < 1e-4] = True  # scattered bright specks
    return implant


@pytest.mark.parametrize("shape", [(32, 48, 48), (60, 64, 80), (128, 128, 128)])
def test_edt_field_matches_oracle(gpu, shape):
    rng = np.random.default_rng(sum(shape))
    implant = _rod_implant(shape, rng)
    cyl = generate_cylinder_mask(shape[1], shape[2])
    _say("edt field", shape)
    want = E.edt_field(implant, cyl)
    assert np.array_equal(edt.generate_edt_field(implant, cyl), want)
    assert np.array_equal(edt.generate_edt_field(implant), want)  # default cylinder mask


def test_device_entries_match_host_entries(gpu):
    rng = np.random.default_rng(1000)
    L = capi.lib()
    shape = (20, 36, 44)
    implant = _rod_implant(shape, rng)
    cyl = generate_cylinder_mask(36, 44).astype(np.uint8)
    data = np.ascontiguousarray(~implant, dtype=np.uint8)
    bufs = [hip.DeviceBuffer.from_array(a) for a in (data, implant.astype(np.uint8), cyl)]
    n = data.size
    sq = hip.DeviceBuffer(4 * n)
    fl = hip.DeviceBuffer(4 * n)
    q = hip.DeviceBuffer(2 * n)
    ws = hip.DeviceBuffer(L.mxb_edt_workspace_bytes(*shape))
    st = hip.Stream()
    capi.check(L.mxb_device_edt(bufs[0].ptr, *shape, sq.ptr, fl.ptr, ws.ptr, st.handle))
    capi.check(L.mxb_device_edt_field(bufs[1].ptr, *shape, bufs[2].ptr, q.ptr, ws.ptr, st.handle))
    st.synchronize()
    assert np.array_equal(sq.to_array(np.uint32, shape).astype(np.uint64), E.edt_sq(data))
    assert np.array_equal(fl.to_array(np.float32, shape), E.edt(data))
    assert np.array_equal(q.to_array(np.uint16, shape), E.edt_field(implant, cyl != 0))
    for b in bufs + [sq, fl, q, ws]:
        b.free()


def test_edt_field_large_host_copies(gpu):
    """A volume whose host copies go through the pinned staging chunks (136 MB
    in, 272 MB out): the host entry equals the device entry bit for bit."""
    rng = np.random.default_rng(1100)
    shape = (520, 512, 512)
    implant = _rod_implant(shape, rng)
    cyl = generate_cylinder_mask(512, 512).astype(np.uint8)
    _say("edt field staged", shape)
    host = edt.generate_edt_field(implant, cyl)
    L = capi.lib()
    dm = hip.DeviceBuffer.from_array(implant.astype(np.uint8))
    dc = hip.DeviceBuffer.from_array(cyl)
    dq = hip.DeviceBuffer(2 * implant.size)
    ws = hip.DeviceBuffer(L.mxb_edt_workspace_bytes(*shape))
    capi.check(L.mxb_device_edt_field(dm.ptr, *shape, dc.ptr, dq.ptr, ws.ptr, None))
    hip.synchronize()
    assert np.array_equal(host, dq.to_array(np.uint16, shape))
    for b in (dm, dc, dq, ws):
        b.free()


# Enough lines for the lane-per-line passes (65536 along y, along z, or both),
# ragged rows, one to four 1024-voxel pieces per row, value and position bits
# that do and do not share a word.
WIDE = [(300, 5, 257), (5, 300, 257), (270, 265, 250), (70, 9, 1030), (33, 40, 2500), (17, 23, 4096), (64, 1025, 65),
        (1200, 70, 1000)]


@pytest.mark.parametrize("case", range(len(WIDE)))
@pytest.mark.parametrize("kind", ["sparse", "dense", "planes", "late"])
def test_edt_many_lines(gpu, case, kind):
    """Few and many sites, equal parabolas all along y and z (the stack holds
    the whole line), and a near site after a long rise (it pops all of it)."""
    shape = WIDE[case]
    rng = np.random.default_rng(1100 + case)
    data = np.ones(shape, bool)
    if kind == "sparse":
        data[rng.random(shape) < 2e-5] = False
    elif kind == "dense":
        data[rng.random(shape) < 0.05] = False
    elif kind == "planes":
        data[:, :, shape[2] // 3] = False
    else:
        y, z = np.meshgrid(np.arange(shape[1]), np.arange(shape[0]))
        x = np.clip(shape[2] // 2 - (y + z) // 2, 0, shape[2] - 1)  # sites move off as y and z grow
        data[z, y, x] = False
        data[-1, -1, :] = False
    data.flat[rng.integers(data.size)] = False
    _say("edt many lines", shape, kind)
    assert np.array_equal(edt.edt_sq(data).astype(np.uint64), E.edt_sq(data))
    if kind == "sparse" and data.size < 20_000_000:
        cyl = generate_cylinder_mask(shape[1], shape[2])
        assert np.array_equal(edt.edt(data), E.edt(data))
        assert np.array_equal(edt.generate_edt_field(~data, cyl), E.edt_field(~data, cyl))


def test_edt_many_lines_without_sites(gpu):
    assert np.all(edt.edt_sq(np.ones((260, 258, 256), bool)) == edt.EDT_NONE)


# A lane per line along y (65536 lines) or along z (131072 lines).
LANES = [(300, 37, 257), (9, 330, 410), (257, 9, 256)]


@pytest.mark.parametrize("case", range(len(LANES)))
@pytest.mark.parametrize("kind", ["noise", "some planes", "some lines", "late gap", "early gap", "just near", "columns"])
def test_edt_of_near_sites(gpu, case, kind):
    """Lines whose sites are near everywhere, up to the farthest distance that
    still counts as near and one more; beside empty lines in one wave; and with
    a gap late or early in the line.  Squares, distances and the field."""
    shape = LANES[case]
    nz, ny, nx = shape
    rng = np.random.default_rng(1300 + case)
    data = np.ones(shape, bool)
    if kind == "noise":
        data[rng.random(shape) < 0.4] = False
    elif kind == "some planes":
        data[rng.random(nz) < 0.4] = False
    elif kind == "some lines":
        data[np.broadcast_to(rng.random((nz, 1, nx)) < 0.3, shape)] = False
    elif kind == "late gap":
        data[rng.random(shape) < 0.5] = False
        data[:, 3 * ny // 4:, nx // 3:] = True
        data[4 * nz // 5:] = True
    elif kind == "early gap":
        data[rng.random(shape) < 0.5] = False
        data[: nz // 3, : ny // 2, 5:] = True
    elif kind == "just near":
        data[3::9 if case % 2 else 11, ::10, ::3] = False
    else:
        data[:, ::9, ::2] = False
    data.flat[rng.integers(data.size)] = False
    _say("edt near sites", shape, kind)
    want = E.edt_sq(data)
    assert np.array_equal(edt.edt_sq(data).astype(np.uint64), want)
    assert np.array_equal(edt.edt(data), E.edt(data))
    cyl = generate_cylinder_mask(ny, nx)
    assert np.array_equal(edt.generate_edt_field(~data, cyl), E.edt_field(~data, cyl))


@pytest.mark.parametrize("kind", ["sparse", "rod", "planes"])
def test_edt_lanes_along_z_distances_and_field(gpu, kind):
    """The lane-per-line pass along z writing distances and the field."""
    for shape in [(9, 330, 410), (33, 300, 451)]:
        rng = np.random.default_rng(1400)
        if kind == "rod":
            implant = _rod_implant(shape, rng)
        else:
            implant = rng.random(shape) < 1e-4
            if kind == "planes":
                implant[:, :, shape[2] // 3] = True
        implant.flat[rng.integers(implant.size)] = True
        _say("edt lanes along z", shape, kind)
        cyl = generate_cylinder_mask(shape[1], shape[2])
        assert np.array_equal(edt.edt(~implant), E.edt(~implant))
        assert np.array_equal(edt.generate_edt_field(implant, cyl), E.edt_field(implant, cyl))


# Short lines along z that look outward: about a run of 8 and of 16, the 16 or 32
# positions looked at one by one, several turns of a block's waves, the longest.
SCAN_DEPTHS = [1, 7, 16, 17, 33, 48, 65, 128, 129, 150, 257, 496, 512]


@pytest.mark.parametrize("n", SCAN_DEPTHS)
def test_edt_scan_of_far_sites(gpu, n):
    """Sites far from most of a line: one, a plane, two planes, a slanted
    plane, a cone, a corner under a plane, sparse sites; ragged last block."""
    ny, nx = 9, 71
    z, y, x = np.ogrid[:n, :ny, :nx]
    rng = np.random.default_rng(1500 + n)
    masks = {
        "one": (z == n // 3) & (y == 4) & (x == 50),
        "plane": (z == n // 2) & (y >= 0) & (x >= 0),
        "ends": ((z == 0) | (z == n - 1)) & (y >= 0) & (x > 30),
        "slanted": (np.abs(x * 1.0 - z * nx / n) < 1) & (y >= 0),
        "cone": (y - 4) ** 2 + (x - 35) ** 2 <= (0.4 * nx * z / n) ** 2,
        "corner": ((z == 0) & (y >= 0) & (x >= 0)) | ((y == 0) & (x == 0) & (z >= 0)),
        "sparse": rng.random((n, ny, nx)) < 2e-4,
        "late": (z >= n - 2) & (x % 5 == 0) & (y >= 0),
    }
    for kind, implant in masks.items():
        implant = np.array(np.broadcast_to(implant, (n, ny, nx)))
        implant.flat[rng.integers(implant.size)] |= kind == "sparse"
        _say("edt scan", n, kind)
        assert np.array_equal(edt.edt_sq(~implant).astype(np.uint64), E.edt_sq(~implant)), kind
        if kind in ("one", "cone", "sparse"):
            cyl = generate_cylinder_mask(ny, nx)
            assert np.array_equal(edt.edt(~implant), E.edt(~implant)), kind
            assert np.array_equal(edt.generate_edt_field(implant, cyl), E.edt_field(implant, cyl)), kind


# Offsets from a corner whose squared distance has a float32 root that depends on
# the last bit of the reciprocal root: of all up to 2^24, those four.
@pytest.mark.parametrize("far", [(12, 74, 2873), (1, 520, 3629), (1, 565, 3745), (1, 2508, 3057)])
def test_edt_root_where_the_reciprocal_decides(gpu, far):
    """8259749, 13440042, 14344251 and 15635314: distances to one corner site."""
    _say("edt root", far)
    data = np.ones(tuple(f + 1 for f in far), dtype=bool)
    data[0, 0, 0] = False
    z, y, x = np.ogrid[:data.shape[0], :data.shape[1], :data.shape[2]]
    want = np.sqrt((z * z + y * y + x * x).astype(np.float32))
    got = edt.edt(data)
    assert got[far] == want[far]
    assert np.array_equal(got, want)
