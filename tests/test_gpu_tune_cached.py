"""The autotuner on grids whose spectrum is kept in cache and whose column tiles
are 16 wide (csrc/fft_kernels.hpp, spec_cached; csrc/tune.cpp): decisions timed on
other kernels are not taken, and tuned variants keep both, with the built-in
kernels' results bit for bit."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (256, 256, 256)  # 75 MB of spectrum, 129 columns: cached, 16-column tiles in y and z


def _tune(cdn, tmp_path, lines, shape):
    d = tmp_path / "cudadecon_amd"
    d.mkdir(parents=True, exist_ok=True)
    (d / "tune_gfx950_v2.txt").write_text("".join(l + "\n" for l in lines))
    old = os.environ.get("XDG_CACHE_HOME")
    os.environ["XDG_CACHE_HOME"] = str(tmp_path)
    try:
        return cdn.autotune([shape], reps=1, use_cache=True)
    finally:
        if old is None:
            del os.environ["XDG_CACHE_HOME"]
        else:
            os.environ["XDG_CACHE_HOME"] = old


def _case(shape):
    kr, kz = np.arange(17) / 32.0, np.fft.fftfreq(33)
    tab = np.exp(-2 * np.pi ** 2 * ((1.5 * kr[:, None]) ** 2 + (3.0 * kz[None, :]) ** 2)).astype(np.complex64)
    ks = tuple(np.float32(v) for v in (32.0 / shape[2], 32.0 / shape[1], 33.0 / shape[0]))
    return tab, ks, np.random.default_rng(5).poisson(30.0, shape).astype(np.float32)


def _run(cdn, tab, ks, raw, n=4):
    e = cdn.RLEngine(raw.shape, tab, ks)
    e.set_raw(raw)
    lam, _ = e.iterate(n)
    x = e.get()
    e.close()
    return x, lam


def test_decisions_of_other_kernels_are_not_taken(cdn, tmp_path):
    """Lines as written for such a grid before it ran cached, narrow kernels."""
    g = "x".join(map(str, SHAPE))
    cdn.autotune_clear()
    rep = _tune(cdn, tmp_path, [f"256 x {g} 0 256 -1 -1 0 0 0", f"256 yz {g} 8 0 1 0 0 0 0"], SHAPE)
    print(rep, flush=True)
    (e,) = rep["lengths"]
    assert "ms" in e["x"] and "ms" in e["columns"]  # timed, not read
    v = cdn.fft_variant(256)
    assert v is None or v["cols"] != 8
    cdn.autotune_clear()


# (shape, the decision file's lines): columns that leave the tile's shape alone
# and ones that change it, x lines, both, and a 2048-point y pass in 16 columns
CASES = [
    (SHAPE, ["256 xc {g} 0 0 -1 -1 0 0 0", "256 yzcn {g} 0 0 1 0 0 0 0"]),
    (SHAPE, ["256 xc {g} 0 0 -1 -1 0 0 0", "256 yzcn {g} 32 0 -1 -1 0 0 0"]),
    ((64, 128, 128), ["64 zn {g} 0 0 1 -1 0 0 4", "128 x {g} 0 0 -1 -1 0 0 0", "128 yn {g} 0 0 1 -1 0 0 0"]),
    ((64, 2048, 512), ["64 z {g} 0 0 -1 -1 0 0 0", "2048 yn {g} 0 0 1 -1 0 0 0", "512 x {g} 0 0 -1 -1 0 0 0"]),
]


@pytest.mark.parametrize("shape,lines", CASES)
def test_column_variants_keep_the_results(cdn, tmp_path, shape, lines):
    tab, ks, raw = _case(shape)
    cdn.autotune_clear()
    x0, lam0 = _run(cdn, tab, ks, raw)
    rep = _tune(cdn, tmp_path, [l.format(g="x".join(map(str, shape))) for l in lines], shape)
    print(shape, [e["chosen"] for e in rep["lengths"]], flush=True)
    for e in rep["lengths"]:
        assert all("cached" in e[k] for k in ("x", "columns") if k in e)  # every line was read
    assert any(cdn.fft_variant(n) for n in shape)
    x1, lam1 = _run(cdn, tab, ks, raw)
    assert np.array_equal(x1, x0) and np.array_equal(lam1, lam0)
    cdn.autotune_clear()


def test_x_variant_keeps_the_results_to_rounding(cdn, tmp_path):
    """Other dot-product blocks, as without a cached spectrum."""
    tab, ks, raw = _case(SHAPE)
    g = "x".join(map(str, SHAPE))
    cdn.autotune_clear()
    x0, lam0 = _run(cdn, tab, ks, raw)
    _tune(cdn, tmp_path, [f"256 xc {g} 0 256 -1 -1 0 0 0", f"256 yzcn {g} 0 0 -1 -1 0 0 0"], SHAPE)
    assert cdn.fft_variant(256)["xthreads"] == 256
    x1, lam1 = _run(cdn, tab, ks, raw)
    assert np.abs(x1 - x0).max() <= 1e-5 * np.abs(x0).max()
    assert np.abs(lam1 - lam0).max() <= 1e-9
    b = cdn.Batch([SHAPE] * 2, tab, [ks] * 2)
    for i in range(2):
        b.set_raw(i, raw)
    for mode in ("graph", "grouped_graph"):
        b.run(4, mode)
        assert np.abs(b.get(1) - x0).max() <= 1e-5 * np.abs(x0).max(), mode
    b.close()
    cdn.autotune_clear()
