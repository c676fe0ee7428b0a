"""Copies between host and device at the edges of their sizes and from several
threads (csrc/hostcopy.cpp): downloads go through the pinned buffers from 2 MB on
(4.5 MB on a stream made for the call), uploads from 16 MB on, in chunks of a quarter of the copy (1 to 16 MB, four
buffers; 32 MB and two buffers from 512 MB on); a download below 16 MB that finds
the buffers taken goes through the runtime.

A zero-angle deskew is a copy with the last column padded, so every result is
bitwise its input."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _copy(cdn, im):
    got = cdn.deskew(im, 0.0, 0.3, 0.104, pad_val=-7.0)
    nx = im.shape[2]
    return got.shape == im.shape and np.array_equal(got[..., : nx - 1], im[..., : nx - 1]) and \
        bool(np.all(got[..., nx - 1:] == np.float32(-7.0)))


# floats per volume: (nz, ny, nx) around each size, partial last chunks among them
SIZES = [(2, 511, 513), (2, 512, 512), (3, 419, 421), (9, 256, 512 - 1), (9, 256, 512), (7, 419, 421), (4, 1024, 1024 - 1), (4, 1024, 1024), (5, 911, 931),
         (17, 997, 1013), (128, 1024, 1024 - 1), (128, 1024, 1024), (131, 1019, 1021)]


@pytest.mark.parametrize("shape", SIZES, ids=lambda s: f"{4 * s[0] * s[1] * s[2] / MB:.2f}MB")
def test_round_trips_at_the_edges_of_sizes(cdn, shape):
    print("host copy", shape, flush=True)
    im = np.random.default_rng(shape[2]).standard_normal(shape, np.float32)
    assert _copy(cdn, im)


@pytest.mark.parametrize("shape", [(64, 64, 96), (64, 64, 128), (64, 96, 128), (64, 128, 192), (64, 192, 256)],
                         ids=lambda s: f"{4 * s[0] * s[1] * s[2] / MB:.2f}MB")
def test_staged_stacks_come_back(cdn, shape):
    """On an engine's own stream: X_0 is the stack that was staged."""
    print("host copy, engine", shape, flush=True)
    im = np.random.default_rng(shape[2]).uniform(0, 100, shape).astype(np.float32)
    e = cdn.RLEngine(shape, np.ones((9, 12), np.complex64), (0.2, 0.2, 0.2))
    e.set_raw(im)
    assert np.array_equal(e.get(), im)
    e.close()


def test_threads_fetch_side_by_side(cdn):
    """Eight threads with results of 3 to 15 MB and one with 24 MB: each gets its
    own data whichever way its copies go."""
    shapes = [(z, 256, 512) for z in (6, 10, 13, 18, 22, 25, 28, 30)] + [(48, 256, 512)]
    ims = [np.random.default_rng(i).standard_normal(s, np.float32) for i, s in enumerate(shapes)]
    bad = []

    def work(im):
        for k in range(6):
            if not _copy(cdn, im):
                bad.append((im.shape, k))

    print("host copies from", len(ims), "threads", flush=True)
    th = [threading.Thread(target=work, args=(im,)) for im in ims]
    for t in th:
        t.start()
    for t in th:
        t.join(100)
    assert not any(t.is_alive() for t in th) and not bad
