"""FP32 passes on rows of any alignment: the direct-load form with 4-byte loads
against the register-ring form (bit for bit) and the oracle, where its groups,
segments and stores have edges: 64 lines exactly, one more, a last group that
overlaps the one before, lines shorter than a tile, several segments."""
import numpy as np
import pytest

import oracle
from maxibone_amd import capi
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
