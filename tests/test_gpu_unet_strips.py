"""Shapes at the edges of the convolution's row strips and column tiles and
of the weight gradient's segments, against the bf16 CPU oracle (the bounds of
test_gpu_unet.py: bfloat16 accuracy of activations and gradients)."""
import sys

import numpy as np
import pytest

from common import product, rel_l2
from unet_oracle import LAYERS, UNetOracle, offsets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w", [(1, 8, 8), (3, 8, 136), (1, 104, 72), (1, 152, 24), (2, 56, 64)])
def test_unet_strips(n, h, w):
    print("unet", n, h, w)
    sys.stdout.flush()
    net = product().UNet(seed=21)
    p = net.get_params()
    wo, bo, _ = offsets()
    rng = np.random.default_rng(22)
    for l, (ci, co, _) in enumerate(LAYERS):
        p[bo[l]:bo[l] + co] = (rng.standard_normal(co) * 0.05).astype(np.float32)
    net.set_params(p)
    x = rng.standard_normal((n, 3, h, w)).astype(np.float32)
    t = (0.5 * x[:, 0] - 0.3 * x[:, 1]).astype(np.float32)
    ref = UNetOracle(p, bf16=True)
    assert rel_l2(net.forward(x), ref.forward(x)) < 1e-2
    loss, g = net.loss_grad(x, t)
    lr, gr = ref.loss_grad(x, t)
    assert abs(loss - lr) <= 1e-2 * abs(lr)
    for l, (ci, co, _) in enumerate(LAYERS):
        sl = slice(wo[l], bo[l] + co)
        if np.max(np.abs(gr[sl])) > 0:
            assert rel_l2(g[sl], gr[sl]) < 5e-2, l


@pytest.mark.parametrize("n,h,w", [(512, 56, 8), (1024, 24, 8), (64, 56, 8)])
def test_unet_strips_of_several_rows(n, h, w):
    """Batches so large that the convolutions' waves walk strips of several
    rows and the weight gradient's workgroups whole images.  Rows per wave of
    512 x 56 rows: 12 (five strips, the last of 8 rows), 6 at half resolution
    (the last of 4), 12 and 3 at a quarter (the last of 2), 1 at an eighth; of
    1024 x 24 rows: 12 at each of 24, 12, 6 and 3 rows.  64 x 56 rows split the
    weight gradient within an image: chunks of 7 and, at a quarter, 4 of 14
    rows.  The sums of a forward
    pass do not depend on the split: the batch gives the bits of its images
    alone."""
    print("unet, strips of several rows", n, h, w)
    sys.stdout.flush()
    net = product().UNet(seed=23)
    p = net.get_params()
    wo, bo, _ = offsets()
    rng = np.random.default_rng(24)
    for l, (ci, co, _) in enumerate(LAYERS):
        p[bo[l]:bo[l] + co] = (rng.standard_normal(co) * 0.05).astype(np.float32)
    net.set_params(p)
    x = rng.standard_normal((n, 3, h, w)).astype(np.float32)
    t = (0.5 * x[:, 0] - 0.3 * x[:, 1]).astype(np.float32)
    ref = UNetOracle(p, bf16=True)
    y = net.forward(x)
    loss, g = net.loss_grad(x, t)
    assert np.array_equal(y[:3], net.forward(np.ascontiguousarray(x[:3])))
    assert np.array_equal(y[-3:], net.forward(np.ascontiguousarray(x[-3:])))
    assert rel_l2(y, ref.forward(x)) < 1e-2
    lr, gr = ref.loss_grad(x, t)
    assert abs(loss - lr) <= 1e-2 * abs(lr)
    for l, (ci, co, _) in enumerate(LAYERS):
        sl = slice(wo[l], bo[l] + co)
        if np.max(np.abs(gr[sl])) > 0:
            assert rel_l2(g[sl], gr[sl]) < 5e-2, l


@pytest.mark.parametrize("copies", [512, 1024, 4096])
def test_unet_batches_of_many_rows(copies):
    """More image rows than the 65536 workgroups of a grid's second dimension:
    69632 and 139264, half of them after pooling; and so many images (forward
    only).  A batch of copies of 17 images gives their outputs' bits and, the scale 2 / pixels being a power
    of two smaller, their gradient up to the fp32 sums over the partials: at
    most 17408 / 4 terms one after the other, 2.6e-4 of the terms' magnitude."""
    print("unet, many rows", copies)
    sys.stdout.flush()
    net = product().UNet(seed=3)
    rng = np.random.default_rng(25)
    x = rng.standard_normal((17, 3, 8, 8)).astype(np.float32)
    t = (0.5 * x[:, 0] - 0.3 * x[:, 1]).astype(np.float32)
    y, (loss, g) = net.forward(x), net.loss_grad(x, t)
    xs, ts = np.tile(x, (copies, 1, 1, 1)), np.tile(t, (copies, 1, 1))
    assert np.array_equal(net.forward(xs), np.tile(y, (copies, 1, 1)))
    if copies > 1024:
        return
    ls, gs = net.loss_grad(xs, ts)
    assert abs(ls - loss) <= 1e-6 * loss
    assert rel_l2(gs, g) < 1e-3
