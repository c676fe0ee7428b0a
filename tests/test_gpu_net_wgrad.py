"""Weight gradients of the warm-start network at the edges of their tiles
(csrc/net_kernels.hip, k_wgrad and k_wgrad_in1): chunks of 64 and 128 voxels of
x, products over 32 voxels, pieces of at least 8 rows of y, planes outside the
volume.  Against the FP64 oracle (oracle/net.py) with the tolerances of the
other gradient tests: the backward tensors are BF16, so per layer 3e-2 relative
L2 to the gradient of the same BF16 forward, and a cosine of 0.995 to the exact
one."""
import numpy as np
import pytest

from oracle import net as N

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 4, 4, 4),      # one voxel at the coarsest level
    (3, 8, 12, 132),   # full size 128 + 4, half size 64 + 2, three samples
    (1, 8, 36, 260),   # two chunks and a remainder
    (2, 16, 68, 64),   # pieces of y with a remainder
    (1, 12, 8, 28),    # less than one product of 32 at every level
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_weight_gradients_at_tile_edges(cdn, shape):
    print("wgrad", shape, flush=True)
    rng = np.random.default_rng(7)
    p = N.he_init(1)
    w_off, b_off, h, _ = N.layout()
    for l in range(5):
        p[b_off[l]:b_off[l] + N.COUT[l]] = 0.05 + 0.05 * rng.random(N.COUT[l])
    p[h:h + 16] = 0.2 * rng.standard_normal(16)
    p = p.astype(np.float32)
    raw = rng.gamma(2.0, 50.0, shape).astype(np.float32)
    tgt = (raw * rng.uniform(0.5, 1.5, shape)).astype(np.float32)
    loss, g = cdn.WarmNet(params=p).loss_grad(raw, tgt)
    loss_b, gb, _, _ = N.loss_grad(p.astype(np.float64), raw, tgt, bf=True)
    _, ge, _, _ = N.loss_grad(p.astype(np.float64), raw, tgt)
    assert abs(loss - loss_b) <= 1e-2 * loss_b
    for l in range(5):
        w = slice(w_off[l], w_off[l] + 27 * N.CIN[l] * N.COUT[l])
        assert np.linalg.norm(g[w] - gb[w]) <= 3e-2 * np.linalg.norm(gb[w]), l
    cos = float(g @ ge / (np.linalg.norm(g) * np.linalg.norm(ge)))
    assert cos >= 0.995


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_bias_gradients_are_the_sums_of_the_backward_tensors(cdn, shape):
    """The same kernels' 28th tap.  Against the FP64 sum of the very BF16 tensor
    that the kernel read: a chain of at most 64 products of 32 voxels in FP32 at
    these sizes, then FP64, so (64 + 32) 2^-24 < 1e-5 of the absolute sum."""
    print("bias grad", shape, flush=True)
    rng = np.random.default_rng(8)
    p = N.he_init(2)
    w_off, b_off, h, _ = N.layout()
    p[h:h + 16] = 0.2 * rng.standard_normal(16)
    raw = rng.gamma(2.0, 50.0, shape).astype(np.float32)
    tgt = (raw * rng.uniform(0.5, 1.5, shape)).astype(np.float32)
    net = cdn.WarmNet(params=p.astype(np.float32))
    _, g = net.loss_grad(raw, tgt)
    for l in range(5):
        pre = net.fetch("dPre%d" % (l + 1)).reshape(-1, N.COUT[l]).astype(np.float64)
        got = g[b_off[l]:b_off[l] + N.COUT[l]]
        assert np.all(np.abs(got - pre.sum(0)) <= 1e-5 * np.abs(pre).sum(0)), l
