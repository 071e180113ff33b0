"""The network on a grid whose weight-gradient partials exceed what is held for all
layers at once: each layer is then reduced before the next one's partials take its
place (device memory of one layer's), with the gradients of the small grid."""
import ctypes as C

import numpy as np
import pytest

from oracle import convnet as cn

pytestmark = pytest.mark.gpu

CIN, COUT, DIL = 9, 3, (1, 2, 4, 1)
SMALL, LARGE, AT = (32, 32, 32), (128, 256, 256), (91, 140, 213)   # AT: place of the small grid in the large one


def problem(rng):
    """Zero biases, and input and target zero outside the middle 8^3 of SMALL: the
    receptive field (8 points a side) stays inside, so the same data anywhere in a
    larger grid has the same gradients, times the quotient of the grids' sizes."""
    p = np.zeros(cn.NL * cn.LAYER_P, dtype=np.float32)
    for l in range(cn.NL):
        ci, co = (CIN if l == 0 else cn.CH), (COUT if l == cn.NL - 1 else cn.CH)
        W = np.zeros((27, cn.CH, cn.CH))
        W[:, :co, :ci] = rng.uniform(-1, 1, (27, co, ci)) * np.sqrt(6.0 / (27 * ci))
        p[l * cn.LAYER_P:l * cn.LAYER_P + cn.LAYER_W] = W.reshape(-1)
    x, t = np.zeros(SMALL + (CIN,), np.float32), np.zeros(SMALL + (COUT,), np.float32)
    x[12:20, 12:20, 12:20] = rng.standard_normal((8, 8, 8, CIN))
    t[12:20, 12:20, 12:20] = rng.standard_normal((8, 8, 8, COUT))
    return p, x, t


def embed(a, grid=LARGE, at=AT):
    b = np.zeros(grid + a.shape[3:], np.float32)
    b[tuple(slice(o, o + n) for o, n in zip(at, SMALL))] = a
    return b.reshape(-1, a.shape[3])


def free_memory():
    """hipMemGetInfo of the runtime the library is linked against."""
    from igap4_amd import _lib
    fr, tot = C.c_size_t(), C.c_size_t()
    assert _lib.lib().hipMemGetInfo(C.byref(fr), C.byref(tot)) == 0
    return fr.value


def test_gradients_and_memory(igap):
    """Against the same network on the small grid, which the oracle pins elsewhere: the
    ratio of the sizes is 256, so every value and every BF16 rounding is the same on
    both grids and only the order of the FP32 sums over the points differs (13,824 points
    that are not zero: 13824^(1/2) 6e-8 = 7e-6 at most).  (The oracle's own FP64 sums
    round a few activations of this little data to other BF16 values, 2e-3 of layer
    0's gradient.)"""
    from igap4_amd import warmstart
    p, x, t = problem(np.random.default_rng(11))
    ratio = np.prod(LARGE) // np.prod(SMALL)
    with warmstart.WarmStartNet(SMALL, CIN, COUT, DIL) as net:
        net.set_params(p)
        loss_ref, g_ref = net.gradients(x.reshape(-1, CIN), t.reshape(-1, COUT))
    before = free_memory()
    with warmstart.WarmStartNet(LARGE, CIN, COUT, DIL) as net:
        used = before - free_memory()
        net.set_params(p)
        loss, g = net.gradients(embed(x), embed(t))
        loss2 = net.train_step(embed(x), embed(t), 0.0)
        loss3, g3 = net.gradients(embed(x), embed(t))
    V = int(np.prod(LARGE))
    need = V * (8 * 32 + 4 * (CIN + 2 * COUT)) + 4 * 27 * 256 * (V // 512)   # activations, fields, one layer's partials
    print(f"  {used / 1e6:.0f} MB for {need / 1e6:.0f}")
    assert used < need + (64 << 20)
    assert loss == loss2 == loss3 and np.array_equal(g, g3)
    assert abs(loss * ratio - loss_ref) < 1e-5 * loss_ref
    for l in range(cn.NL):
        o = l * cn.LAYER_P
        for sl in (slice(o, o + cn.LAYER_W), slice(o + cn.LAYER_W, o + cn.LAYER_P)):
            err = np.linalg.norm(g[sl] * ratio - g_ref[sl]) / max(np.linalg.norm(g_ref[sl]), 1e-30)
            print(f"  layer {l} rel err {err:.2e}")
            assert err < 1e-5


def test_remainder_of_the_partials(igap):
    """10125 partials of 512 points are 39 rounds of 256 and a shorter one: the same data
    in an early round and in the last one (points from 5111808 on, so x >= 3944) has
    the same gradients but for the order of the sums, as above."""
    from igap4_amd import warmstart
    p, x, t = problem(np.random.default_rng(12))
    grid = (4000, 36, 36)
    out = []
    with warmstart.WarmStartNet(grid, CIN, COUT, DIL) as net:
        net.set_params(p)
        for at in ((100, 1, 3), (3960, 2, 2)):
            out.append(net.gradients(embed(x, grid, at), embed(t, grid, at)))
    (loss, g), (loss2, g2) = out
    assert abs(loss - loss2) < 1e-5 * loss
    for l in range(cn.NL):
        o = l * cn.LAYER_P
        for sl in (slice(o, o + cn.LAYER_W), slice(o + cn.LAYER_W, o + cn.LAYER_P)):
            assert np.linalg.norm(g[sl] - g2[sl]) < 1e-5 * np.linalg.norm(g[sl])
