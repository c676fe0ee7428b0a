"""The kernels with 64-bit addresses, for z filters whose planes (and transforms
whose slabs) span 2 GiB and more, on small stacks: csrc/fft_kernels.hpp,
WideAddresses, held by the calling thread.  The same arithmetic in another form,
so the built-in lengths give the buffer kernels' results bit for bit; run-time
compiled ones may contract differently and are held to the FP64 oracle's
tolerance."""
import contextlib
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4


@contextlib.contextmanager
def _wide(cdn):
    L = cdn.lib()
    obj = (ctypes.c_char * 8)()
    L["_ZN3cdn13WideAddressesC1Ev"](ctypes.byref(obj))
    try:
        yield
    finally:
        L["_ZN3cdn13WideAddressesD1Ev"](ctypes.byref(obj))


def _ra():
    kr, kz = np.arange(9) / 16.0, np.fft.fftfreq(12)
    return np.exp(-2 * np.pi ** 2 * ((1.5 * kr[:, None]) ** 2 + (2.0 * kz[None, :]) ** 2)).astype(np.complex64)


def _3d():
    fz, fy, fx = np.fft.fftfreq(12), np.fft.fftfreq(16), np.arange(9) / 16.0
    return np.exp(-2 * np.pi ** 2 * ((2.0 * fz[:, None, None]) ** 2 + (1.5 * fy[None, :, None]) ** 2 +
                                     (1.5 * fx[None, None, :]) ** 2)).astype(np.complex64)


# every built-in z length; 33 columns of 96 and 192 run as one run-time compiled tile; 50 is compiled at run time
SHAPES = [(64, 16, 64), (64, 16, 400), (96, 16, 64), (128, 16, 64), (128, 16, 400), (192, 16, 64), (256, 16, 64),
          (256, 16, 400), (384, 8, 64), (512, 8, 64), (768, 8, 64), (810, 8, 64), (1024, 4, 64), (2048, 4, 64),
          (50, 16, 64)]


@pytest.mark.parametrize("kind", ["averaged", "3-D"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_wide_z_filters_give_the_same(cdn, orc, shape, kind):
    nz, ny, nx = shape
    tab = _ra() if kind == "averaged" else _3d()
    ks = tuple(np.float32(v) for v in (0.99913 * 16.0 / nx, 16.0 / ny, 12.0 / nz))
    raw = np.random.default_rng(nz).poisson(30.0, shape).astype(np.float32)

    def run():
        e = cdn.RLEngine(shape, tab, ks)
        e.set_raw(raw)
        lam, _ = e.iterate(3)
        out = [e.get(), lam]
        e.close()
        b = cdn.Batch([shape] * 2, tab, [ks] * 2)
        for i in range(2):
            b.set_raw(i, raw)
        for mode in ("grouped", "grouped_graph"):
            b.run(3, mode)
            out += [b.get(1), b.lambdas(1, 3)]
        b.close()
        return out

    print("wide addresses", shape, kind, flush=True)
    a = run()
    with _wide(cdn):
        w = run()
    if nz % 5 == 0 and nz != 810:
        dims = (9, 1, 12) if kind == "averaged" else (9, 16, 12)
        ref, _ = orc.rl_ba(raw, orc.otf_interp(tab, dims, (nx, ny, nz), ks), 3)
        for x in (w[0], w[2], w[4]):
            assert np.abs(x - ref).max() <= TOL * np.abs(ref).max()
    else:
        for x, y in zip(a, w):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("shape", [(64, 96, 64), (256, 128, 64), (192, 256, 64), (384, 512, 64), (768, 810, 16),
                                   (1024, 64, 32), (64, 2048, 64), (2048, 16, 32)],
                         ids=lambda s: "x".join(map(str, s)))
def test_wide_transforms_give_the_same(cdn, shape):
    v = np.random.default_rng(shape[0]).uniform(0, 100, shape).astype(np.float32)
    print("wide transforms", shape, flush=True)
    s = cdn.fft_r2c(v)
    b = cdn.fft_c2r(s, shape[2])
    with _wide(cdn):
        sw = cdn.fft_r2c(v)
        bw = cdn.fft_c2r(s, shape[2])
    assert np.array_equal(s, sw) and np.array_equal(b, bw)
