"""What preparing a run-time compiled length builds (csrc/jit.cpp): the kernels
that its stacks launch, not those for slabs of 2 GiB and more, which are a module
of their own, compiled at first need."""
import os
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTH = 245  # used by no other test: its code is not in this process yet
# k_col<N, inverse, false>, and of the averaged kind k_z_filter<N, 1, false>, k_z_ragged<N, persistent, 1, false>
WIDE = re.compile(rb"k_colILi\d+ELb[01]ELb0E|k_z_filterILi\d+ELi1ELb0E|k_z_raggedILi\d+ELb[01]ELi1ELb0E")


def test_preparing_a_length_leaves_out_the_wide_slab_kernels(cdn, tmp_path):
    shape = (64, LENGTH, 64)
    kr, kz = np.arange(17) / 32.0, np.fft.fftfreq(33)
    tab = np.exp(-2 * np.pi ** 2 * ((1.5 * kr[:, None]) ** 2 + (3.0 * kz[None, :]) ** 2)).astype(np.complex64)
    ks = tuple(np.float32(v) for v in (32.0 / shape[2], 32.0 / shape[1], 33.0 / shape[0]))
    old = os.environ.get("XDG_CACHE_HOME")
    os.environ["XDG_CACHE_HOME"] = str(tmp_path)
    try:
        print("run-time length", LENGTH, flush=True)
        e = cdn.RLEngine(shape, tab, ks)
        e.set_raw(np.random.default_rng(1).poisson(30.0, shape).astype(np.float32))
        e.iterate(3)
        assert np.isfinite(e.get()).all()
        e.close()
    finally:
        if old is None:
            del os.environ["XDG_CACHE_HOME"]
        else:
            os.environ["XDG_CACHE_HOME"] = old
    files = list((tmp_path / "cudadecon_amd").glob(f"fft_{LENGTH}_*.hsaco"))
    assert files
    for f in files:
        names = f.read_bytes().split(b"\x7fELF")[0]
        assert b"k_z_filter" in names and not WIDE.search(names), f.name
