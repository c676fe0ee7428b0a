"""The OTF's support bound where its last ky row has a number beyond 2^31: a long
table and a small ky scale, so that every row lies inside (csrc/decon.cpp,
OtfDev::params).  Against the FP64 oracle's filter of the whole spectrum;
tolerance as the other filter tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,ky", [(3000, 1.2e-6), (2100, 1.1e-6), (3000, 4e-6), (9, 1.2e-6)])
def test_small_ky_scale_keeps_every_row(cdn, orc, nr, ky):
    nz, ny, nx = 64, 96, 64
    rng = np.random.default_rng(nr)
    # smooth in the radius: its FP32 rounding (3000 * 2^-24) then moves no value by more than 1e-7
    tab = (np.linspace(1.0, 0.6, nr)[:, None] *
           (rng.uniform(0.2, 1.0, 4) + 1j * rng.uniform(-0.5, 0.5, 4))[None, :]).astype(np.complex64)
    ks = tuple(np.float32(v) for v in (0.99913 * 2 * (nr - 1) / nx, ky, 4.0 / nz))
    v = rng.uniform(0, 100, (nz, ny, nx)).astype(np.float32)
    print("support limits", nr, ky, flush=True)
    ref = orc.filt(v.astype(np.float64), orc.otf_interp(tab, (nr, 1, 4), (nx, ny, nz), ks))
    got = cdn.filter_volume(v, tab, ks)
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
