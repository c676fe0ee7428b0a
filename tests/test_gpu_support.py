"""The OTF's support bound in the y transforms and the z filter: rows outside
it are neither stored, filtered nor read (csrc/fft_kernels_dev.hpp,
support_ky), against the FP64 oracle's filter of the whole spectrum.

The table is random up to its last radial sample, so a row cut too early
shows in the result; tolerance as the other filter tests (FP32 transforms
against FP64).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# k-scales relative to the last radial sample at Nyquist in x and y
SCALES = {
    "covers all": (0.3, 0.3),      # no column cut
    "corners": (1.0, 1.0),         # data and PSF sampled alike
    "half": (2.1, 1.9),            # whole kx columns outside
    "narrow in y": (0.9, 7.3),
    "narrow in x": (11.7, 0.8),
    "centre only": (40.1, 40.3),   # a few columns and rows left
    "constant in x": (0.0, 1.2),   # no bound
}


@pytest.mark.parametrize("nr", [2, 9])
@pytest.mark.parametrize("scale", SCALES, ids=lambda s: s.replace(" ", "-"))
@pytest.mark.parametrize("shape", [(64, 96, 192), (96, 256, 64), (128, 64, 128), (45, 63, 70)],
                         ids=lambda s: "x".join(map(str, s)))
def test_filter_with_bounded_support_matches_oracle(cdn, orc, shape, scale, nr):
    nz, ny, nx = shape
    rng = np.random.default_rng(nr * 1000 + nz)
    tab = (rng.uniform(0.2, 1.0, (nr, 12)) + 1j * rng.uniform(-0.5, 0.5, (nr, 12))).astype(np.complex64)
    sx, sy = SCALES[scale]
    # a factor off 1 keeps every radius away from the last sample itself
    ks = tuple(np.float32(v) for v in (0.99913 * sx * 2 * (nr - 1) / nx, 1.00071 * sy * 2 * (nr - 1) / ny, 12.0 / nz))
    v = rng.uniform(0, 100, shape).astype(np.float32)
    H = orc.otf_interp(tab, (nr, 1, 12), (nx, ny, nz), ks)
    for conj in (False, True):
        print("support", shape, scale, nr, conj, flush=True)
        ref = orc.filt(v.astype(np.float64), H, conj=conj)
        got = cdn.filter_volume(v, tab, ks, conj=conj)
        assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()


# tiles of 16 columns (csrc/fft_kernels.hip, y_narrow and z_narrow): exactly one
# tile, one column more, several with a remainder, the last count with narrow z
# tiles and the first without
@pytest.mark.parametrize("shape", [(64, 128, 30), (128, 64, 32), (256, 128, 64), (128, 256, 315), (64, 128, 320)],
                         ids=lambda s: "x".join(map(str, s)))
def test_narrow_tiles_match_oracle(cdn, orc, shape):
    nz, ny, nx = shape
    rng = np.random.default_rng(nx)
    tab = (rng.uniform(0.2, 1.0, (9, 12)) + 1j * rng.uniform(-0.5, 0.5, (9, 12))).astype(np.complex64)
    ks = tuple(np.float32(v) for v in (0.99913 * 16 / nx, 1.00071 * 16 / ny, 12.0 / nz))
    v = rng.uniform(0, 100, shape).astype(np.float32)
    print("narrow", shape, flush=True)
    ref = orc.filt(v.astype(np.float64), orc.otf_interp(tab, (9, 1, 12), (nx, ny, nz), ks))
    got = cdn.filter_volume(v, tab, ks)
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
