"""The z filter of a 3-D OTF table, through buffers at 64 and 128 points and by
addresses elsewhere (csrc/fft_kernels_dev.hpp, zf_buf), in tiles of 16 and more
columns: iterations and grouped batches against the FP64 oracle, and batches
bitwise against single engines.  z lengths with a factor of 5 leave out the
last: there the 3-D kind's interpolation has always been contracted differently
in the grouped kernel (differences of 1e-6 relative).  Tolerance as the other
iteration tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _table():
    fz, fy, fx = np.fft.fftfreq(12), np.fft.fftfreq(16), np.arange(9) / 16.0
    t = -2 * np.pi ** 2 * ((2.0 * fz[:, None, None]) ** 2 + (1.5 * fy[None, :, None]) ** 2 +
                           (1.5 * fx[None, None, :]) ** 2)
    return (np.exp(t) * np.exp(-2j * np.pi * 0.02 * fz[:, None, None])).astype(np.complex64)


# (nz, ny, nx): narrow tiles up to 160 columns
SHAPES = [(64, 24, 60), (64, 12, 400), (128, 24, 60), (128, 12, 400), (256, 12, 64), (256, 12, 400), (96, 12, 64),
          (810, 6, 40), (50, 24, 64)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_iterations_and_batches_with_a_3d_table(cdn, orc, shape):
    nz, ny, nx = shape
    tab = _table()
    ks = tuple(np.float32(v) for v in (0.99913 * 16.0 / nx, 16.0 / ny, 12.0 / nz))
    rng = np.random.default_rng(nz + nx)
    raw = rng.poisson(30.0, shape).astype(np.float32)
    print("3-D table", shape, flush=True)
    e = cdn.RLEngine(shape, tab, ks)
    e.set_raw(raw)
    lam, _ = e.iterate(4)
    x = e.get()
    e.close()
    ref, _ = orc.rl_ba(raw, orc.otf_interp(tab, (9, 16, 12), (nx, ny, nz), ks), 4)
    assert np.abs(x - ref).max() <= TOL * np.abs(ref).max()
    bitwise = nz % 5 != 0
    b = cdn.Batch([shape] * 2, tab, [ks] * 2)
    for i in range(2):
        b.set_raw(i, raw)
    for cap in (0, 8):
        b.set_grid_cap(cap)
        b.run(4, "grouped")
        for i in range(2):
            assert np.abs(b.get(i) - ref).max() <= TOL * np.abs(ref).max(), cap
            if bitwise:
                assert np.array_equal(b.get(i), x) and np.array_equal(b.lambdas(i, 4), lam), cap
    b.close()
