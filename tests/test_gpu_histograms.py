"""Histogram and combination kernels at the sizes where their shapes change: ragged rows,
volumes that start off a 16-byte boundary, table widths from 1 to the most
bins, radii around the annulus edges, centres off the volume, and value ranges
whose bin edges fall on whole numbers.  Counts and combined fields equal the oracle's."""
import numpy as np
import pytest

from maxibone_amd import capi, hip
from oracle import fields as F

pytestmark = pytest.mark.gpu


def _at(a, shift):
    """A device copy of `a` that starts `shift` bytes after an aligned address."""
    buf = hip.DeviceBuffer(a.nbytes + 64)
    hip.check(hip.rt().hipMemcpy(buf.ptr + shift, np.ascontiguousarray(a).ctypes.data, a.nbytes, hip.H2D))
    return buf


AXIS = [  # shape, z_offset, Nz, Nr, bins, centre, range, byte shift, distinct values
    ((3, 1, 1), 0, 3, 1, 1, (0, 0), (1.0, 65535.0), 0, None),
    ((5, 7, 9), 0, 5, 40, 3, (30, -20), (0.0, 65535.0), 2, None),
    ((70, 9, 130), 5, 60, 70, 256, (4, 65), (1.0, 40000.0), 0, None),
    ((33, 40, 61), 0, 33, 50, 4096, (20, 30), (1.0, 40000.0), 6, None),
    ((40, 64, 72), 0, 40, 16, 4096, (32, 36), (13333.0, 26666.0), 0, None),
    ((40, 64, 72), 0, 40, 17, 4097, (31, 36), (0.1, 60000.7), 0, None),
    ((9, 33, 264), 0, 9, 150, 8192, (16, 132), (65000.0, 1000.0), 0, None),
    ((9, 33, 264), 0, 9, 150, 8192, (16, 132), (1.0, 65535.0), 8, None),
    ((300, 30, 16), 0, 300, 20, 512, (15, 8), (1.0, 65535.0), 0, 2),
    ((2, 1300, 24), 0, 2, 700, 64, (650, 12), (1.0, 65535.0), 0, None),
    ((4, 40, 40), 0, 4, 30, 100, (20, 20), (500.0, 500.0), 0, None),
]


@pytest.mark.parametrize("case", range(len(AXIS)))
def test_axis_histograms_at_edges(gpu, case):
    shape, z_off, Nz, Nr, vb, centre, vrange, shift, distinct = AXIS[case]
    print("axis histograms", AXIS[case], flush=True)
    rng = np.random.default_rng(900 + case)
    if distinct:
        vox = (rng.integers(0, distinct, shape) * 30000).astype(np.uint16)
    else:
        vox = rng.integers(0, 65536, shape, dtype=np.uint16)
        vox[rng.random(shape) < 0.1] = 13333
    sizes = (shape[2], shape[1], Nz, Nr)
    bins = [rng.integers(0, 3, (n, vb)).astype(np.uint64) for n in sizes]
    with np.errstate(all="ignore"):
        if vrange[0] < vrange[1]:
            want = F.axis_histograms(vox, z_off, *[b.copy() for b in bins], centre, vrange)
        else:
            want = bins  # no value lies in the range, or the bin is 0/0
    L = capi.lib()
    dv = _at(vox, shift)
    db = [hip.DeviceBuffer.from_array(b) for b in bins]
    ws = hip.DeviceBuffer(L.mxb_histogram_workspace_bytes(*shape))
    capi.check(L.mxb_device_axis_histograms(dv.ptr + shift, *shape, z_off, *(b.ptr for b in db), Nz, Nr, vb,
                                            centre[0] % 2**64, centre[1] % 2**64, *vrange, ws.ptr, None))
    for b, w, n in zip(db, want, sizes):
        assert np.array_equal(b.to_array(np.uint64, (n, vb)), w)


def _smooth(shape, top=65535.0):
    z, y, x = (np.linspace(-1, 1, n) if n > 1 else np.zeros(1) for n in shape)
    r = np.sqrt(y[:, None] ** 2 + x[None, :] ** 2)
    f = top * np.exp(-3 * r)[None] * (1 + 0.2 * z[:, None, None]) / 1.2
    return np.clip(f, 0, 65535).astype(np.uint16)


FIELD = [  # voxel shape, field shape, (field bins, voxel bins), voxel range, field range, noisy field
    ((1, 1, 1), (1, 1, 1), (1, 1), (0.0, 65535.0), (0.0, 65535.0), False),
    ((20, 40, 37), (20, 40, 37), (2048, 4096), (1.0, 40000.0), (1.0, 65535.0), False),
    ((33, 50, 71), (17, 25, 36), (2048, 4096), (1.0, 40000.0), (1.0, 65535.0), False),
    ((33, 50, 71), (22, 33, 47), (500, 5000), (0.1, 60000.7), (100.5, 30000.25), False),
    ((40, 64, 96), (10, 16, 24), (1024, 256), (1.0, 65535.0), (1.0, 65535.0), False),
    ((40, 64, 96), (5, 8, 12), (7, 3), (1.0, 65535.0), (20000.0, 50000.0), False),
    ((36, 44, 52), (3, 4, 4), (300, 1000), (1.0, 65535.0), (1.0, 65535.0), False),     # boxes above the limit
    ((24, 24, 24), (24, 24, 24), (60, 32768), (1.0, 65535.0), (1.0, 65535.0), False),  # one row per group
    ((24, 24, 24), (24, 24, 24), (60, 32769), (1.0, 65535.0), (1.0, 65535.0), False),  # no row fits
    ((24, 24, 24), (24, 24, 24), (2048, 32768), (1.0, 65535.0), (1.0, 65535.0), False),
    ((24, 24, 24), (24, 24, 24), (2049, 32768), (1.0, 65535.0), (1.0, 65535.0), False),  # groups beyond the limit
    ((40, 40, 40), (40, 40, 40), (2048, 4096), (1.0, 65535.0), (1.0, 65535.0), True),  # every brick meets most groups
    ((40, 40, 40), (20, 20, 20), (2048, 4096), (1.0, 65535.0), (1.0, 65535.0), True),
    ((10, 12, 14), (20, 12, 30), (64, 64), (1.0, 65535.0), (1.0, 65535.0), False),     # field finer than the voxels
    ((24, 24, 24), (24, 24, 24), (64, 64), (1.0, 65535.0), (65535.0, 1.0), False),     # bins fall with the value
    ((600, 9, 10), (600, 9, 10), (64, 4096), (30000.0, 30100.0), (60000.0, 60001.0), False),
]


@pytest.mark.parametrize("case", range(len(FIELD)))
def test_field_histogram_at_edges(gpu, case):
    vshape, fshape, nbins, vrange, frange, noisy = FIELD[case]
    print("field histogram", FIELD[case], flush=True)
    rng = np.random.default_rng(950 + case)
    vox = np.clip(rng.normal(30000, 9000, vshape), 0, 65535).astype(np.uint16)
    vox[rng.random(vshape) < 0.1] = 0
    fld = rng.integers(0, 65536, fshape, dtype=np.uint16) if noisy else _smooth(fshape)
    fld[rng.random(fshape) < 0.05] = 0
    init = rng.integers(0, 5, nbins).astype(np.uint64)
    want = F.field_histogram(vox, fld, init.copy(), vrange, frange)
    L = capi.lib()
    dv, df, db = hip.DeviceBuffer.from_array(vox), hip.DeviceBuffer.from_array(fld), hip.DeviceBuffer.from_array(init)
    ws = hip.DeviceBuffer(L.mxb_histogram_workspace_bytes(*vshape))
    capi.check(L.mxb_device_field_histogram(dv.ptr, *vshape, df.ptr, *fshape, db.ptr, *nbins, *vrange, *frange,
                                            ws.ptr, None))
    assert np.array_equal(db.to_array(np.uint64, nbins), want)


COMBINE = [  # shape, byte shift of the fields, cylinder: None, "all", "none", "disc", "random"
    ((1, 1, 2), 0, None), ((3, 5, 7), 2, "random"), ((70, 9, 11), 0, "disc"), ((2, 33, 64), 6, "none"),
    ((5, 40, 64), 0, "all"), ((4, 200, 211), 2, "disc"), ((300, 16, 128), 0, "random"),
]


@pytest.mark.parametrize("case", range(len(COMBINE)))
def test_combine_at_edges(gpu, case):
    shape, shift, kind = COMBINE[case]
    print("combine", COMBINE[case], flush=True)
    rng = np.random.default_rng(980 + case)
    g = rng.integers(0, 60000, shape, dtype=np.uint16)
    e = rng.integers(0, 65536, shape, dtype=np.uint16)
    g.flat[0], e.flat[0], g.flat[-1], e.flat[-1] = 59999, 0, 0, 65535
    cyl = {None: None, "all": np.ones(shape[1:], bool), "none": np.zeros(shape[1:], bool),
           "disc": (np.add.outer((np.arange(shape[1]) - shape[1] / 2) ** 2, (np.arange(shape[2]) - shape[2] / 2) ** 2)
                    < (min(shape[1:]) / 2) ** 2), "random": rng.random(shape[1:]) > 0.5}[kind]
    want = F.combine_fields(g, e, np.ones(shape[1:], bool) if cyl is None else cyl)
    L = capi.lib()
    dg, de, out = _at(g, shift), _at(e, shift), hip.DeviceBuffer(g.nbytes + 64)
    dc = None if cyl is None else hip.DeviceBuffer.from_array(cyl.astype(np.uint8))
    ws = hip.DeviceBuffer(L.mxb_combine_workspace_bytes())
    capi.check(L.mxb_device_combine_fields(dg.ptr + shift, de.ptr + shift, *shape, None if dc is None else dc.ptr,
                                           out.ptr, ws.ptr, None))
    assert np.array_equal(out.to_array(np.uint16, shape), want)


LONG = [  # voxel shape, field shape: tables of more words than the workspace's fixed part
    ((1, 1, 140000), (1, 1, 140000)), ((2, 3, 200000), (2, 3, 200000)), ((150000, 2, 3), (75000, 1, 2)),
    ((3, 131200, 1), (3, 43733, 1)),
]


@pytest.mark.parametrize("case", range(len(LONG)))
def test_field_histogram_of_long_axes_stays_in_its_workspace(gpu, case):
    vshape, fshape = LONG[case]
    print("field histogram, long axis", LONG[case], flush=True)
    rng = np.random.default_rng(990 + case)
    vox = rng.integers(0, 65536, vshape, dtype=np.uint16)
    fld = rng.integers(0, 65536, fshape, dtype=np.uint16)
    nbins, vrange, frange = (64, 128), (1.0, 65535.0), (1.0, 65535.0)
    want = F.field_histogram(vox, fld, np.zeros(nbins, np.uint64), vrange, frange)
    L = capi.lib()
    size, guard = L.mxb_histogram_workspace_bytes(*vshape), 1 << 20
    ws = hip.DeviceBuffer.from_array(np.full(size + guard, 0xA5, np.uint8))
    dv, df = hip.DeviceBuffer.from_array(vox), hip.DeviceBuffer.from_array(fld)
    db = hip.DeviceBuffer.from_array(np.zeros(nbins, np.uint64))
    capi.check(L.mxb_device_field_histogram(dv.ptr, *vshape, df.ptr, *fshape, db.ptr, *nbins, *vrange, *frange,
                                            ws.ptr, None))
    assert np.array_equal(db.to_array(np.uint64, nbins), want)
    assert np.all(ws.to_array(np.uint8, (size + guard,))[size:] == 0xA5)


SLABS = [  # shape, Nr, bins, centre: slabs a few rows or columns thick, also seen from afar
    ((3000, 1, 300), 200, 16, (0, 150)), ((9000, 2, 70), 80, 5, (1, 3)), ((700, 3, 2000), 2000, 64, (1, 1000)),
    ((5000, 90, 1), 60, 9, (45, 0)), ((2500, 2, 2), 500, 7, (-300, 40)), ((40, 1, 3000), 4000, 300, (900, 10)),
    ((66000, 1, 9), 12, 3, (0, 4)), ((300, 1300, 2), 700, 33, (650, 1)),
]


@pytest.mark.parametrize("case", range(len(SLABS)))
def test_axis_histograms_of_thin_slabs(gpu, case):
    """Equal voxels, so that every counter of a ring takes all of its pixels in
    all of a block's layers, and voxels of two values."""
    shape, Nr, vb, centre = SLABS[case]
    for top in (1, 2):
        print("thin slab", SLABS[case], top, flush=True)
        vox = (np.random.default_rng(70 + case).integers(0, top, shape) * 20000 + 30000).astype(np.uint16)
        sizes = (shape[2], shape[1], shape[0], Nr)
        want = F.axis_histograms(vox, 0, *[np.zeros((n, vb), np.uint64) for n in sizes], centre, (1.0, 65535.0))
        L = capi.lib()
        dv = hip.DeviceBuffer.from_array(vox)
        db = [hip.DeviceBuffer.from_array(np.zeros((n, vb), np.uint64)) for n in sizes]
        ws = hip.DeviceBuffer(L.mxb_histogram_workspace_bytes(*shape))
        capi.check(L.mxb_device_axis_histograms(dv.ptr, *shape, 0, *(b.ptr for b in db), shape[0], Nr, vb,
                                                centre[0] % 2**64, centre[1] % 2**64, 1.0, 65535.0, ws.ptr, None))
        for b, w, n in zip(db, want, sizes):
            assert np.array_equal(b.to_array(np.uint64, (n, vb)), w)


MANY = [  # voxel shape, field shape, bins, noisy field
    ((150, 150, 130), (150, 150, 130), (2048, 4096), False),  # several thousand bricks
    ((232, 232, 240), (232, 232, 240), (400, 4096), True),    # a block's list of bricks fills more than once
    ((8000, 400, 1), (8000, 400, 1), (300, 512), False),      # bricks enlarged to fit their table
    ((40, 45, 70), (9, 11, 8), (64, 4096), False),            # uneven boxes of up to 5 x 5 x 9
    ((61, 77, 83), (30, 38, 41), (2048, 4096), True),         # of 2 or 3 a side
    ((61, 77, 83), (20, 51, 82), (2048, 256), False),         # of 3 or 4, 1 or 2, and 1 or 2
]


@pytest.mark.parametrize("case", range(len(MANY)))
def test_field_histogram_of_many_bricks_and_uneven_boxes(gpu, case):
    vshape, fshape, nbins, noisy = MANY[case]
    print("field histogram", MANY[case], flush=True)
    rng = np.random.default_rng(1050 + case)
    vox = np.clip(rng.normal(30000, 9000, vshape), 0, 65535).astype(np.uint16)
    fld = rng.integers(0, 65536, fshape, dtype=np.uint16) if noisy else _smooth(fshape)
    vrange = frange = (1.0, 65535.0)
    want = F.field_histogram(vox, fld, np.zeros(nbins, np.uint64), vrange, frange)
    L = capi.lib()
    dv, df = hip.DeviceBuffer.from_array(vox), hip.DeviceBuffer.from_array(fld)
    db = hip.DeviceBuffer.from_array(np.zeros(nbins, np.uint64))
    ws = hip.DeviceBuffer(L.mxb_histogram_workspace_bytes(*vshape))
    capi.check(L.mxb_device_field_histogram(dv.ptr, *vshape, df.ptr, *fshape, db.ptr, *nbins, *vrange, *frange,
                                            ws.ptr, None))
    assert np.array_equal(db.to_array(np.uint64, nbins), want)


FEW = ["none", "one", "two", "four", "rare"]


@pytest.mark.parametrize("noisy", [True, False])
@pytest.mark.parametrize("kind", FEW)
def test_field_histogram_of_voxels_of_few_values(gpu, kind, noisy):
    """Voxels of so few values that they are hashed where others are grouped;
    among them values in places that a sample may miss."""
    vshape, fshape, nbins, vrange = (184, 180, 186), (92, 90, 93), (2048, 4096), (1.0, 40000.0)
    print("field histogram of few values", kind, noisy, flush=True)
    rng = np.random.default_rng(1070)
    values = {"none": [0, 50000], "two": [900, 40000], "four": [0, 1, 900, 901]}.get(kind, [900])
    vox = np.array(values, np.uint16)[rng.integers(0, len(values), vshape)]
    if kind == "rare":
        vox[90, 91:99] = rng.integers(0, 65536, (8, 186))
        vox[0, 0, 0] = vox[-1, -1, -1] = 40000
    fld = rng.integers(0, 65536, fshape, dtype=np.uint16) if noisy else _smooth(fshape)
    want = F.field_histogram(vox, fld, np.zeros(nbins, np.uint64), vrange, (1.0, 65535.0))
    L = capi.lib()
    dv, df = hip.DeviceBuffer.from_array(vox), hip.DeviceBuffer.from_array(fld)
    db = hip.DeviceBuffer.from_array(np.zeros(nbins, np.uint64))
    ws = hip.DeviceBuffer(L.mxb_histogram_workspace_bytes(*vshape))
    capi.check(L.mxb_device_field_histogram(dv.ptr, *vshape, df.ptr, *fshape, db.ptr, *nbins, *vrange, 1.0, 65535.0,
                                            ws.ptr, None))
    assert np.array_equal(db.to_array(np.uint64, nbins), want)


def test_field_histogram_of_more_than_2_31_bins(gpu):
    """Voxel bins from 2^31 on count where they lie (17 GB of bins, of which
    the few that count are read back)."""
    vb, vox = (1 << 31) + 64, np.array([[[1, 65535, 32768, 65534, 65535]]], np.uint16)
    fld = np.full((1, 1, 5), 7, np.uint16)
    L = capi.lib()
    db = hip.DeviceBuffer(8 * vb)
    db.fill_bytes(0)
    dv, df = hip.DeviceBuffer.from_array(vox), hip.DeviceBuffer.from_array(fld)
    ws = hip.DeviceBuffer(L.mxb_histogram_workspace_bytes(*vox.shape))
    print("field histogram of", vb, "bins", flush=True)
    capi.check(L.mxb_device_field_histogram(dv.ptr, *vox.shape, df.ptr, *fld.shape, db.ptr, 1, vb, 1.0, 65535.0, 1.0,
                                            65535.0, ws.ptr, None))

    def count(i):
        one = np.empty(1, np.uint64)
        hip.check(hip.rt().hipMemcpy(one.ctypes.data, db.ptr + 8 * i, 8, hip.D2H))
        return int(one[0])

    def bin_of(v):
        return int(np.floor(np.float64(vb - 1) * ((np.float64(v) - 1.0) / 65534.0)))

    assert bin_of(65535) == vb - 1
    assert [count(bin_of(v)) for v in (1, 32768, 65534, 65535)] == [1, 1, 1, 2]
    assert count((1 << 31) - 1) == 0
    db.free()
