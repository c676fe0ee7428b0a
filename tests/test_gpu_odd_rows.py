"""Stacks with an odd number of rows (ny nz): the last line of the x passes
holds one row only, and the row after it belongs to somebody else.

LRcore takes its rows through buffers at the lengths that split through LDS
(csrc/fft_kernels_dev.hpp, lr_buf); the missing row is left out by the vector
offset, which alone takes part in a buffer's range check.  49 rows leave one row
to the last workgroup at every x length here (2, 4, 16 and 24 rows per
workgroup).  Against the FP64 oracle, and bitwise in a batch whose odd stacks
lie back to back with others of the same x length, where a row too many would
land in the next stack's spectrum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4  # FP32 against the FP64 oracle, as the other iteration tests


def _table():
    kr, kz = np.arange(17) / 32.0, np.fft.fftfreq(33)
    return np.exp(-2 * np.pi ** 2 * ((1.5 * kr[:, None]) ** 2 + (3.0 * kz[None, :]) ** 2)).astype(np.complex64)


def _kscale(shape):
    return tuple(np.float32(v) for v in (32.0 / shape[2], 32.0 / shape[1], 33.0 / shape[0]))


# built-in lengths with one, two and eight lines per workgroup, run-time
# compiled ones (100, 600), and 256, whose lines keep addresses
@pytest.mark.parametrize("nx", [64, 96, 128, 192, 810, 2048, 100, 600, 256])
def test_odd_row_counts(cdn, orc, nx):
    tab = _table()
    shapes = [(7, 7, nx), (7, 7, nx), (3, 5, nx), (7, 9, nx), (4, 7, nx)]
    ks = [_kscale(s) for s in shapes]
    rng = np.random.default_rng(nx)
    raws = [rng.poisson(30.0, s).astype(np.float32) for s in shapes]
    refs, lams = [], []
    for s, k, r in zip(shapes, ks, raws):
        print("odd rows, single", s, flush=True)
        e = cdn.RLEngine(s, tab, k)
        e.set_raw(r)
        lam, _ = e.iterate(5)
        x = e.get()
        e.close()
        ref, _ = orc.rl_ba(r, orc.otf_interp(tab, (17, 1, 33), s[::-1], k), 5)
        assert np.abs(x - ref).max() <= TOL * np.abs(ref).max(), s
        refs.append(x)
        lams.append(lam)
    b = cdn.Batch(shapes, tab, ks, nstreams=2)
    for i, r in enumerate(raws):
        b.set_raw(i, r)
    for mode, parts in (("sequential", 1), ("grouped", 1), ("grouped_graph", 1), ("grouped_graph", 2)):
        print("odd rows, batch", nx, mode, parts, flush=True)
        b.set_partitions(parts)
        b.run(5, mode)
        for i in range(len(shapes)):
            assert np.array_equal(b.get(i), refs[i]), (mode, parts, i)
            assert np.array_equal(b.lambdas(i, 5), lams[i]), (mode, parts, i)
    b.close()
