"""FP32 passes on rows of any alignment: the direct-load form with 4-byte loads
against the register-ring form (bit for bit) and the oracle, where its groups,
segments and stores have edges: 64 lines exactly, one more, a last group that
overlaps the one before, lines shorter than a tile, several segments."""
import numpy as np
import pytest

import oracle
from maxibone_amd import capi, hip
from maxibone_amd.helpers import gauss_kernel

pytestmark = pytest.mark.gpu

SHAPES = [(3, 64, 65), (5, 65, 67), (17, 127, 129), (2, 200, 70), (70, 66, 301), (1, 65, 131), (40, 129, 68),
          (33, 403, 66), (9, 30, 99), (300, 70, 65)]


@pytest.mark.parametrize("case", range(len(SHAPES)))
@pytest.mark.parametrize("sigma", [0.6, 3.0, 15.0])
def test_rows_of_any_alignment(gpu, monkeypatch, case, sigma):
    shape = SHAPES[case]
    print("any alignment", shape, sigma, flush=True)
    rng = np.random.default_rng(1200 + case)
    mask = (rng.random(shape) > 0.97).astype(np.uint8)
    k = gauss_kernel(sigma).astype(np.float32)
    got = [capi.diffusion(mask, k, 3, precision="fp32", u16=True, f32=True),
           capi.diffusion(mask, k, 2, precision="fp32", u16=True, f32=False)]
    monkeypatch.setenv("MXB_PASS_KERNEL", "ring")
    want = [capi.diffusion(mask, k, 3, precision="fp32", u16=True, f32=True),
            capi.diffusion(mask, k, 2, precision="fp32", u16=True, f32=False)]
    assert np.array_equal(got[0][0], want[0][0]) and np.array_equal(got[0][1], want[0][1])
    assert np.array_equal(got[1][0], want[1][0])
    u, _ = oracle.diffusion_f32(mask, k, 3)
    assert np.abs(got[0][1] - u).max() <= 1e-5


@pytest.mark.parametrize("sigma", [0.9, 1.9, 2.9, 3.9, 5.9, 7.9, 9.9, 11.9])
@pytest.mark.parametrize("prec", ["fp32_split", "bf16", "fp16"])
def test_fused_pass_steps_of_16_and_32_rows(gpu, prec, sigma):
    """The fused x -> y pass steps by 32 rows where a plane is small enough for
    32-bit offsets, else by 16.  A few columns of mask at the edge of a very
    wide volume (16 rows a step) and of a narrow one (32) give the same values,
    bit for bit, in the columns that the other columns cannot reach; one
    radius of each compiled size."""
    ny, wide, narrow, reps = 41, 1 << 19, 968, 3
    k = gauss_kernel(sigma).astype(np.float32)
    keep = narrow - reps * (len(k) // 2)
    rng = np.random.default_rng(31)
    m = np.zeros((2, ny, wide), np.uint8)
    m[:, :, :keep] = rng.random((2, ny, keep)) > 0.95
    print("fused steps", prec, sigma, flush=True)
    a = capi.diffusion(m, k, reps, precision=prec, u16=True, f32=True)
    b = capi.diffusion(np.ascontiguousarray(m[:, :, :narrow]), k, reps, precision=prec, u16=True, f32=True)
    keep -= len(k) // 2
    assert np.array_equal(a[0][:, :, :keep], b[0][:, :, :keep])
    assert np.array_equal(a[1][:, :, :keep], b[1][:, :, :keep])


@pytest.mark.parametrize("prec, bar", [("fp32_split", 1e-5), ("bf16", 2e-3), ("fp16", 2e-3)])
@pytest.mark.parametrize("shape", [(1, 31, 8), (2, 32, 120), (1, 65, 136), (1, 700, 264), (3, 1, 1024)])
def test_fused_pass_edges(gpu, prec, bar, shape):
    """Rows about one step, strips with a last piece of 8 columns, planes cut
    into several segments, each with the outputs of the last repetition alone
    and together."""
    rng = np.random.default_rng(77)
    m = (rng.random(shape) > 0.95).astype(np.uint8)
    for sigma in (1.2, 4.0, 11.0):
        k = gauss_kernel(sigma).astype(np.float32)
        print("fused edges", prec, shape, sigma, flush=True)
        q, u = capi.diffusion(m, k, 3, precision=prec, u16=True, f32=True)
        ref = oracle.diffusion_f64(m, k.astype(np.float64), 3)
        assert np.abs(u - ref).max() <= bar and np.all(u[m > 0] == 1.0)
        assert np.array_equal(q, capi.diffusion(m, k, 3, precision=prec, u16=True, f32=False)[0])
        assert np.array_equal(u, capi.diffusion(m, k, 3, precision=prec, u16=False, f32=True)[1])


@pytest.mark.parametrize("n", [(4 << 20) - 1, 4 << 20, (4 << 20) + 1, (8 << 20) + 1, (33 << 20) + 5, (70 << 20) + 3])
def test_host_copies(gpu, n):
    """Volumes in host memory about the sizes where the staged copies start,
    end in a part of a piece, and use their ring again; from two threads at
    once.  No repetition: the outputs are the mask's own values."""
    import threading

    print("host copies", n, flush=True)
    m = (np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8) > 100).astype(np.uint8).reshape(1, 1, n)
    out = [None, None]

    def run(i):
        out[i] = capi.diffusion(m, np.ones(1, np.float32), 0, precision="fp32", u16=True, f32=True)

    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for q, u in out:
        assert np.array_equal(u, m.astype(np.float32))
        assert np.array_equal(q, np.where(m, np.uint16(65535), np.uint16(0)))


YX_SHAPES = [(1, 1, 4), (2, 63, 32), (3, 64, 36), (1, 65, 96), (2, 130, 128), (1, 200, 613), (30, 20, 31),
             (1, 3, 1), (5, 129, 1000), (260, 300, 70)]


@pytest.mark.parametrize("sigma", [1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 8.0, 10.0, 12.0, 14.0, 16.0])
def test_fused_fp32_y_and_x(gpu, monkeypatch, sigma):
    """The FP32 form's fused y -> x pass against the register-ring passes, bit
    for bit, one radius of each compiled size: tiles of 64 rows and pairs of 32
    columns exactly, one more and one less, rows of 4-byte and of 16-byte
    pieces, one and several segments, each set of outputs."""
    k = gauss_kernel(sigma).astype(np.float32)
    for i, shape in enumerate(YX_SHAPES):
        print("fused y and x", shape, sigma, flush=True)
        m = (np.random.default_rng(500 + i).random(shape) > 0.96).astype(np.uint8)
        for out in ({"u16": True, "f32": True}, {"u16": True, "f32": False}, {"u16": False, "f32": True}):
            monkeypatch.delenv("MXB_PASS_KERNEL", raising=False)
            got = capi.diffusion(m, k, 2, precision="fp32", **out)
            monkeypatch.setenv("MXB_PASS_KERNEL", "ring")
            want = capi.diffusion(m, k, 2, precision="fp32", **out)
            for a, b in zip(got, want):
                assert (a is None) == (b is None) and (a is None or np.array_equal(a, b))


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_fused_fp32_y_and_x_in_batches(gpu, monkeypatch, prec):
    """The batched form's fused y -> x pass against its separate passes and the
    single-volume form, bit for bit: rows whose last 16-byte piece holds pads,
    rows of one pad less and more than a line, each radius size up to 40."""
    shapes = [(3, 5, 7), (20, 64, 32), (9, 65, 33), (30, 63, 97), (4, 130, 126), (17, 31, 161), (2, 200, 62)]
    sigmas = [2.0, 3.0, 4.0, 5.0, 6.0, 8.0, 10.0]
    rng = np.random.default_rng(9)
    ms = [(rng.random(s) > 0.95).astype(np.uint8) for s in shapes]
    ks = [gauss_kernel(s).astype(np.float32) for s in sigmas]
    print("fused batch", prec, flush=True)
    got = capi.diffusion_batched(ms, ks, 3, precision=prec, u16=True, f32=True)
    monkeypatch.setenv("MXB_XY_FUSED", "0")
    want = capi.diffusion_batched(ms, ks, 3, precision=prec, u16=True, f32=True)
    for i in range(len(ms)):
        assert np.array_equal(got[0][i], want[0][i]) and np.array_equal(got[1][i], want[1][i])
        if prec == "fp32":
            one = capi.diffusion(ms[i], ks[i], 3, precision=prec, u16=True, f32=True)
            assert np.array_equal(got[0][i], one[0]) and np.array_equal(got[1][i], one[1])


@pytest.mark.parametrize("prec", ["fp32", "fp32_exact", "bf16", "fp16", "fp32_split"])
def test_start_from_the_mask(gpu, prec):
    """The start of a diffusion (state and mask bits in one kernel, or two for
    short rows of larger volumes): with a single tap of 1 the result is
    (mask > 0) exactly, for any byte that is not zero, at the edges of a tile of
    32 rows and 128 columns."""
    shapes = [(2, 33, nx) for nx in (1, 7, 31, 32, 33, 95, 96, 127, 128, 129, 300)] + [(70, 80, 95), (5, 1, 640)]
    for i, shape in enumerate(shapes):
        print("start", prec, shape, flush=True)
        rng = np.random.default_rng(40 + i)
        m = (rng.integers(0, 256, shape) * (rng.random(shape) > 0.5)).astype(np.uint8)
        for reps in (1, 3):
            q, u = capi.diffusion(m, np.ones(1, np.float32), reps, precision=prec, u16=True, f32=True)
            assert np.array_equal(u, (m > 0).astype(np.float32)), shape
            assert np.array_equal(q, np.where(m > 0, np.uint16(65535), np.uint16(0))), shape


@pytest.mark.parametrize("prec", ["bf16", "fp16"])
@pytest.mark.parametrize("sigma", [1.0, 3.0, 10.0, 15.0])
def test_pitched_16_bit_rows(gpu, monkeypatch, prec, sigma):
    """16-bit repetitions on rows that are not whole 16-byte pieces run in a
    pitched copy of the state: bit for bit the register-ring passes, at extents
    one from a multiple of 8, of 32 and of 64, with odd and even repetitions
    (either buffer last), and where the pitch does not fit the buffers."""
    k = gauss_kernel(sigma).astype(np.float32)
    for i, shape in enumerate([(20, 33, 65), (9, 64, 63), (65, 31, 127), (3, 129, 130), (40, 100, 33), (7, 9, 9),
                               (2, 3, 1001), (30, 5, 3), (1, 257, 259)]):
        rng = np.random.default_rng(90 + i)
        m = (rng.integers(0, 256, shape) * (rng.random(shape) > 0.95)).astype(np.uint8)
        for reps in (2, 3, 4):
            print("pitched", prec, sigma, shape, reps, flush=True)
            monkeypatch.delenv("MXB_PASS_KERNEL", raising=False)
            got = capi.diffusion(m, k, reps, precision=prec, u16=True, f32=True)
            monkeypatch.setenv("MXB_PASS_KERNEL", "ring")
            want = capi.diffusion(m, k, reps, precision=prec, u16=True, f32=True)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("prec, shape, sigma", [("fp32", (20, 70, 64), 3.0), ("fp32", (9, 65, 67), 10.0),
                                                ("fp32", (40, 33, 30), 15.0), ("bf16", (20, 33, 65), 3.0)])
def test_output_in_a_state_buffer(gpu, prec, shape, sigma):
    """The float output in the state buffer that the separate passes' last
    x-pass does not read (the buffers swap roles each repetition, and once
    more before the 16-bit forms' FP32 repetition) is the output of a buffer
    of its own."""
    n = int(np.prod(shape))
    m = (np.random.default_rng(61).random(shape) > 0.97).astype(np.uint8)
    k = gauss_kernel(sigma).astype(np.float32)
    L = capi.lib()
    dm = hip.DeviceBuffer.from_array(m)
    size = L.mxb_state_bytes(capi.PRECISION[prec], *shape)
    for reps in (1, 2, 3, 4):
        print("output in a state buffer", prec, shape, sigma, reps, flush=True)
        st, own = [hip.DeviceBuffer(size) for _ in range(2)], hip.DeviceBuffer(4 * n)
        free = st[reps % 2] if prec == "fp32" or reps == 1 else st[1 - reps % 2]
        for out in (own, free):
            capi.check(L.mxb_device_diffusion(dm.ptr, *shape, k.ctypes.data, k.size, reps, capi.PRECISION[prec],
                                              st[0].ptr, st[1].ptr, None, out.ptr, None))
            hip.synchronize()
        assert np.array_equal(free.to_array(np.float32, shape), own.to_array(np.float32, shape))


def test_batch_choice_belongs_to_its_passes(gpu, monkeypatch, tmp_path):
    """A plan with the y- and x-passes apart does not take the grid and segment
    that were timed for the fused pass: the file of choices holds one for each,
    and a second plan of one kind takes the first one's."""
    choices = tmp_path / "choices"
    monkeypatch.setenv("MXB_TUNE_FILE", str(choices))
    shape, k = (21, 75, 99), gauss_kernel(2.0).astype(np.float32)
    m = hip.DeviceBuffer.from_array((np.random.default_rng(3).random(shape) > 0.9).astype(np.uint8))
    q = hip.DeviceBuffer(2 * int(np.prod(shape)))
    info = []
    for fused in ("1", "0", "1", "0"):
        monkeypatch.setenv("MXB_XY_FUSED", fused)
        plan = capi.BatchPlan([m.ptr], [shape], [k], 2, outs_u16=[q.ptr])
        info.append(plan.info())
        plan.close()
    keys = [line.split()[0] for line in choices.read_text().splitlines() if "_21x75x99r" in line]
    print(info, keys, flush=True)
    assert len(set(keys)) == 2
    assert info[0] == info[2] and info[1] == info[3]


@pytest.mark.parametrize("pinned", [(True, True), (True, False), (False, True)])
def test_host_copies_of_pinned_memory(gpu, pinned):
    """Masks and outputs in pinned memory, from an address within the
    allocation, and beside pageable ones: the mask's own values, as from
    pageable memory."""
    import ctypes

    n = (33 << 20) + 5
    H = hip.rt()
    H.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    H.hipHostFree.argtypes = [ctypes.c_void_p]
    held = []

    def array(pin, dtype):
        if not pin:
            return np.zeros(n, dtype)
        p, size = ctypes.c_void_p(), n * np.dtype(dtype).itemsize
        hip.check(H.hipHostMalloc(ctypes.byref(p), size + 64, 0))
        held.append(p)
        a = np.frombuffer((ctypes.c_char * size).from_address(p.value + 64), dtype)
        a[:] = 0
        return a

    print("pinned", pinned, flush=True)
    m, q, u = array(pinned[0], np.uint8), array(pinned[1], np.uint16), array(pinned[1], np.float32)
    m[:] = np.random.default_rng(4).random(n) > 0.5
    k = np.ones(1, np.float32)
    capi.check(capi.lib().mxb_diffusion_ex(m.ctypes.data, 1, 1, n, k.ctypes.data, 1, 0, 0, q.ctypes.data, u.ctypes.data, 0))
    assert np.array_equal(u, m.astype(np.float32))
    assert np.array_equal(q, np.where(m, np.uint16(65535), np.uint16(0)))
    del m, q, u
    for p in held:
        hip.check(H.hipHostFree(p))


THIN = [(130, 4, 60), (60, 12, 100), (33, 20, 64), (20, 60, 36), (9, 76, 68), (100, 24, 40), (300, 4, 96)]


@pytest.mark.parametrize("fused", ["1", "0"])
@pytest.mark.parametrize("sigma", [1.0, 4.0, 12.0, 16.0])
def test_thin_volumes_and_separate_passes(gpu, monkeypatch, fused, sigma):
    """Rows of whole 16-byte pieces in thin volumes, whose y lines are shorter or
    longer than 64 positions and leave tiles of 64 rows and rounds of blocks
    part empty, and rows of any alignment, with the y- and x-passes fused and
    apart: bit for bit the register-ring passes, each set of outputs."""
    k = gauss_kernel(sigma).astype(np.float32)
    for i, shape in enumerate(THIN + SHAPES):
        print("thin", shape, sigma, fused, flush=True)
        m = (np.random.default_rng(700 + i).random(shape) > 0.97).astype(np.uint8)
        for out in ({"u16": True, "f32": True}, {"u16": True, "f32": False}, {"u16": False, "f32": True}):
            monkeypatch.delenv("MXB_PASS_KERNEL", raising=False)
            monkeypatch.setenv("MXB_XY_FUSED", fused)
            got = capi.diffusion(m, k, 2, precision="fp32", **out)
            monkeypatch.setenv("MXB_PASS_KERNEL", "ring")
            want = capi.diffusion(m, k, 2, precision="fp32", **out)
            for a, b in zip(got, want):
                assert (a is None) == (b is None) and (a is None or np.array_equal(a, b))
