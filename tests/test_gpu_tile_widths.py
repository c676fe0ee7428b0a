"""Tile widths and the cached build at the lengths that the small cases leave out:
1024 and 2048 points on each axis with a spectrum kept in cache, 2048-point y
columns 16 to a tile (streaming and cached), and 16-column engines against a
batch whose wider stacks make the group's tiles wide.  The same arithmetic
everywhere, so bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(shape, n, seed):
    kr, kz = np.arange(17) / 32.0, np.fft.fftfreq(33)
    tab = np.exp(-2 * np.pi ** 2 * ((1.5 * kr[:, None]) ** 2 + (3.0 * kz[None, :]) ** 2)).astype(np.complex64)
    ks = tuple(np.float32(v) for v in (32.0 / shape[2], 32.0 / shape[1], 33.0 / shape[0]))
    return tab, ks, np.random.default_rng(seed).poisson(30.0, (n,) + shape).astype(np.float32)


def _single(cdn, tab, ks, raw, n=4):
    e = cdn.RLEngine(raw.shape, tab, ks)
    e.set_raw(raw)
    lam, _ = e.iterate(n)
    x = e.get()
    e.close()
    return x, lam


def _spectrum(shape):
    return 8 * shape[0] * shape[1] * ((shape[2] // 2 + 1 + 15) // 16 * 16)


# one stack's spectrum below 32 MB (streaming), all of them above (cached)
@pytest.mark.parametrize("shape,n", [((64, 64, 1024), 2), ((64, 1024, 64), 2), ((1024, 64, 64), 2),
                                     ((16, 64, 2048), 4), ((16, 2048, 64), 3), ((2048, 16, 64), 3)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_cached_long_lines_are_bitwise_the_streaming_ones(cdn, shape, n):
    print("cached long lines", shape, n, flush=True)
    assert _spectrum(shape) < 32 << 20 <= n * _spectrum(shape)
    tab, ks, raw = _case(shape, n, 7)
    m = cdn.RLEngine(shape, tab, ks, stacks=n)
    m.set_raw(raw)
    lam, _ = m.iterate(4)
    b = cdn.Batch([shape] * n, tab, [ks] * n)
    for i in range(n):
        b.set_raw(i, raw[i])
    b.run(4, "grouped")
    for i in (0, n - 1):
        x, l1 = _single(cdn, tab, ks, raw[i])
        assert np.array_equal(m.get_stack(i), x) and np.array_equal(lam[:, i], l1)
        assert np.array_equal(b.get(i), x)
    m.close()
    b.close()


# 16 tiles of 16 columns a plane: 1024 of them (256 MB of spectrum: cached) and
# 1152 (288 MB: streaming); a batch takes these columns 8 to a tile
@pytest.mark.parametrize("nz", [64, 72])
def test_2048_point_columns_16_to_a_tile(cdn, nz):
    shape = (nz, 2048, 480)
    print("2048-point columns", shape, flush=True)
    assert (_spectrum(shape) <= 256 << 20) == (nz == 64) and nz * 16 >= 1024
    tab, ks, raw = _case(shape, 1, 9)
    x, lam = _single(cdn, tab, ks, raw[0], 3)
    b = cdn.Batch([shape], tab, [ks])
    b.set_raw(0, raw[0])
    b.run(3, "grouped")
    assert np.array_equal(b.get(0), x) and np.array_equal(b.lambdas(0, 3), lam)
    b.close()


@pytest.mark.parametrize("shapes", [[(64, 128, 128), (64, 128, 512)], [(128, 64, 128), (128, 256, 512)],
                                    [(256, 128, 64), (256, 128, 400)]],
                         ids=lambda v: "+".join("x".join(map(str, s)) for s in v))
def test_narrow_engines_match_wide_batches(cdn, shapes):
    print("narrow engines, wide batch", shapes, flush=True)
    cases = [_case(s, 1, i) for i, s in enumerate(shapes)]
    tab = cases[0][0]
    b = cdn.Batch(shapes, tab, [c[1] for c in cases])
    for i, c in enumerate(cases):
        b.set_raw(i, c[2][0])
    for cap in (0, 64):
        b.set_grid_cap(cap)
        b.run(4, "grouped")
        for i, c in enumerate(cases):
            x, lam = _single(cdn, tab, c[1], c[2][0])
            assert np.array_equal(b.get(i), x) and np.array_equal(b.lambdas(i, 4), lam), (cap, i)
    b.close()
