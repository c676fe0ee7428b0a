"""Spectra of 32 to 256 MB run the kernels that keep them in cache
(csrc/fft_kernels.hpp, spec_cached), smaller and larger ones the streaming
kernels: the same arithmetic, so a stack gives bitwise the same result and
factors on its own (a small spectrum, streaming) and among others in one
engine (a spectrum inside the range), and so does the grouped batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(shape, n, seed):
    rng = np.random.default_rng(seed)
    kr, kz = np.arange(17) / 32.0, np.fft.fftfreq(33)
    tab = np.exp(-2 * np.pi ** 2 * ((1.5 * kr[:, None]) ** 2 + (3.0 * kz[None, :]) ** 2)).astype(np.complex64)
    ks = tuple(np.float32(v) for v in (32.0 / shape[2], 32.0 / shape[1], 33.0 / shape[0]))
    return tab, ks, rng.poisson(30.0, (n,) + shape).astype(np.float32)


# every built-in length from 64 to 810 on some axis; n stacks bring the spectrum
# above 32 MB
@pytest.mark.parametrize("shape,n", [((64, 128, 128), 8), ((96, 192, 256), 2), ((128, 96, 384), 3), ((192, 64, 512), 3),
                                     ((64, 256, 192), 3), ((256, 64, 96), 6), ((64, 384, 64), 6), ((64, 96, 810), 3)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_cached_spectrum_is_bitwise_the_streaming_one(cdn, shape, n):
    print("cached spectrum", shape, n, flush=True)
    tab, ks, raw = _case(shape, n, 3)
    pitch = (shape[2] // 2 + 1 + 15) // 16 * 16
    one = 8 * shape[0] * shape[1] * pitch
    assert one < 32 << 20 <= n * one
    m = cdn.RLEngine(shape, tab, ks, stacks=n)
    m.set_raw(raw)
    lam, _ = m.iterate(4)
    e = cdn.RLEngine(shape, tab, ks)
    b = cdn.Batch([shape] * n, tab, [ks] * n)
    for i in range(n):
        b.set_raw(i, raw[i])
    b.run(4, "grouped")
    for i in (0, n - 1):
        e.set_raw(raw[i])
        le, _ = e.iterate(4)
        x = e.get()
        assert np.array_equal(m.get_stack(i), x) and np.array_equal(lam[:, i], le)
        assert np.array_equal(b.get(i), x)
