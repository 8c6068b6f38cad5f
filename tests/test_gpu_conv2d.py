"""conv2d implicit GEMM (fp32 MFMA) on the GPU vs the float64 oracle.

Gate: rtol 1e-3 (benchmark configuration) with the registry's atol 1e-3."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import assert_close, launch, ptr, run_registry, seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c,o,r,s,st,pad", [
    (1, 8, 8, 32, 64, 3, 3, 1, 1),       # fast path, one tile
    (2, 9, 7, 64, 64, 3, 3, 1, 1),       # ragged M, borders
    (2, 10, 10, 64, 128, 3, 3, 1, 0),    # valid conv, two N tiles
    (1, 11, 13, 32, 40, 3, 3, 2, 1),     # stride 2, O not a tile multiple
    (3, 6, 6, 64, 64, 1, 1, 1, 0),       # 1x1 = GEMM
    (1, 7, 9, 3, 5, 3, 3, 1, 1),         # generic path (C % 32 != 0)
    (2, 5, 6, 20, 70, 2, 3, 1, 2),       # generic path, pad > filter/2
    (1, 3, 3, 32, 64, 5, 5, 1, 2),       # filter larger than the image interior
])
def test_conv2d_shapes(mb, dev, n, h, w, c, o, r, s, st, pad):
    x = seeded(n * h + c, (n, h, w, c))
    wt = seeded(o * r + s, (o, r, s, c), ("kaiming_normal", r * s * c))
    p = (h + 2 * pad - r) // st + 1
    q = (w + 2 * pad - s) // st + 1
    d_x, d_w = x.to(dev), wt.to(dev)
    d_y = torch.full((n, p, q, o), float("nan"), device=dev)
    launch("mb_launch_conv2d_nhwc_f32", ptr(d_x), ptr(d_w), ptr(d_y), n, h, w, c, o, r, s, st, pad,
           None)
    want = oracle.conv2d_nhwc(x.numpy(), wt.numpy(), st, pad)
    assert_close(d_y.cpu().numpy(), want, 1e-3, 1e-3, f"conv2d {n,h,w,c,o,r,s,st,pad}")


def _random_conv_shapes(n, seed=73):
    """Seeded geometries: channel counts of the fast path (multiples of 32) and
    of the generic one, 1x1 to 5x5 filters, stride 1 or 2, padding 0..2."""
    rng = np.random.default_rng(seed)
    out = []
    while len(out) < n:
        r, s_ = int(rng.choice([1, 3, 5])), int(rng.choice([1, 3, 5]))
        st, pad = int(rng.choice([1, 2])), int(rng.integers(0, 3))
        nb, h, w = int(rng.integers(1, 4)), int(rng.integers(1, 17)), int(rng.integers(1, 17))
        c = int(rng.choice([32, 64, 96, 5, 20]))
        o = int(rng.integers(1, 140))
        if h + 2 * pad < r or w + 2 * pad < s_:
            continue
        out.append((nb, h, w, c, o, r, s_, st, pad))
    return out


@pytest.mark.parametrize("n,h,w,c,o,r,s,st,pad", _random_conv_shapes(10))
def test_conv2d_random_shapes(mb, dev, n, h, w, c, o, r, s, st, pad):
    test_conv2d_shapes(mb, dev, n, h, w, c, o, r, s, st, pad)


def test_conv2d_rejects_bad_geometry(mb, dev):
    from metalbench_amd import native
    lib = native.load()
    d = torch.zeros(16, device=dev)
    assert lib.mb_launch_conv2d_nhwc_f32(ptr(d), ptr(d), ptr(d), 1, 2, 2, 1, 1, 5, 5, 1, 0,
                                         None) == -7
    assert lib.mb_launch_conv2d_nhwc_f32(ptr(d), ptr(d), ptr(d), 1, 2, 2, 1, 1, 1, 1, 0, 0,
                                         None) == -7


@pytest.mark.parametrize("name", ["conv2d", "conv2d_ref"])
def test_conv2d_registry_config(mb, name):
    b, inputs, outs, _ = run_registry(name, seed=0)
    pad = b.meta["model_kwargs"]["padding"]
    want = oracle.conv2d_nhwc(inputs[0].numpy(), inputs[1].numpy(), 1, pad)
    assert_close(outs[0].numpy(), want, b.rtol, b.atol, name)


# The kernel on bf16 term products: chunks of four channels, or elements; one and
# several 16-deep units per wave, many and few tiles, ragged pixels and channels.
@pytest.mark.parametrize("n,h,w,c,o,r,s,st,pad", [
    (24, 60, 61, 4, 8, 1, 1, 1, 0), (24, 60, 61, 3, 65, 3, 3, 1, 1), (23, 60, 60, 20, 66, 2, 3, 1, 1),
    (3, 301, 303, 3, 40, 7, 7, 1, 3), (24, 60, 60, 36, 32, 1, 1, 1, 0), (7, 230, 119, 12, 30, 3, 3, 2, 1),
    (2, 17, 19, 36, 130, 3, 3, 1, 1), (3, 9, 9, 7, 64, 1, 1, 1, 0), (1, 40, 30, 6, 20, 5, 3, 2, 2),
    # K <= 32 (element-wise, unless one unit of whole chunks in the second or fourth round
    # of 256 tiles: 458, 1024 and, further down, 957 of them) and just past it
    (8, 60, 61, 4, 8, 1, 1, 1, 0), (16, 64, 64, 8, 64, 1, 1, 1, 0),
    (24, 60, 61, 5, 65, 3, 3, 1, 1), (24, 50, 50, 11, 64, 1, 3, 1, 0), (24, 50, 51, 20, 40, 1, 1, 1, 0),
    (24, 50, 51, 16, 40, 1, 1, 1, 0), (24, 50, 51, 2, 40, 3, 5, 1, 1),
])
def test_conv2d_split_shapes(mb, dev, n, h, w, c, o, r, s, st, pad):
    """A sum is added up in 6 steps per 16 k (and 3 for the waves' parts), each rounding
    to at worst 2^-23 of a partial sum, which is at most the sum of the products'
    magnitudes; the term products left out are under 2^-26 of each, one more step."""
    x, wt = seeded(n * h + c, (n, h, w, c)), seeded(o * r + s, (o, r, s, c))
    p, q = (h + 2 * pad - r) // st + 1, (w + 2 * pad - s) // st + 1
    d_x, d_w = x.to(dev), wt.to(dev)
    d_y = torch.full((n * p * q * o + 16,), 7.0, device=dev)
    launch("mb_launch_conv2d_nhwc_f32", ptr(d_x), ptr(d_w), ptr(d_y), n, h, w, c, o, r, s, st, pad, None)
    got = d_y[:n * p * q * o].cpu().numpy().reshape(n, p, q, o)
    want = oracle.conv2d_nhwc(x.numpy(), wt.numpy(), st, pad)
    size = oracle.conv2d_nhwc(np.abs(x.numpy()), np.abs(wt.numpy()), st, pad)
    off = np.abs(got - want) / np.where(size > 0, size, 1)
    print("largest error / sum of magnitudes: 2^%.1f" % np.log2(off.max()), flush=True)
    assert off.max() <= (6 * -(-r * s * c // 16) + 4) * 2.0 ** -23
    assert torch.all(d_y[n * p * q * o:] == 7.0)


@pytest.mark.parametrize("n,c", [(24, 4), (24, 3), (24, 5), (1, 4), (1, 3)])
def test_conv2d_values_the_split_cannot_hold(mb, dev, n, c):
    """Infinities, NaN and channels near the smallest normal number."""
    h = w = 60
    x, wt = seeded(1, (n, h, w, c)), seeded(2, (8, 3, 3, c))
    x[0, 5, 7, 1], x[0, 30, 30, 0] = float("inf"), float("nan")
    wt[3] *= 1e-37
    wt[5, 1, 1, 0] = float("-inf")
    d_x, d_w = x.to(dev), wt.to(dev)
    d_y = torch.zeros((n, h, w, 8), device=dev)
    launch("mb_launch_conv2d_nhwc_f32", ptr(d_x), ptr(d_w), ptr(d_y), n, h, w, c, 8, 3, 3, 1, 1, None)
    with np.errstate(all="ignore"):
        want = oracle.conv2d_nhwc(x.numpy(), wt.numpy(), 1, 1)
    xf, wf = np.nan_to_num(x.numpy(), posinf=0, neginf=0), np.nan_to_num(wt.numpy(), posinf=0, neginf=0)
    size = oracle.conv2d_nhwc(np.abs(xf), np.abs(wf), 1, 1)
    got = d_y.cpu().numpy()
    # (a padded tap multiplies zero by the infinite weight in the oracle and in the kernel)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    assert np.all(np.abs(got[fin] - want[fin]) <= (2.0 ** -20 * size)[fin])


@pytest.mark.parametrize("c", [4, 3, 5, 64])
def test_conv2d_small_weights_keep_their_bits(mb, dev, c):
    """A patch that a ReLU left at zero except under one tiny weight: the outputs are
    that product alone, exact up to one rounding (the bound leaves room for one more)."""
    n, h, w, o = 32, 56, 56, 64
    x = torch.zeros((n, h, w, c))
    x[..., 1] = seeded(1, (n, h, w)).clamp_min(0) * 1e30
    wt = seeded(2, (o, 3, 3, c))
    wt[..., 1] = 0.0
    wt[:, 1, 1, 1] = 1.37 * 2.0 ** -torch.arange(100, 100 + o).clamp_max(126).float()
    d_x, d_w = x.to(dev), wt.to(dev)
    d_y = torch.zeros((n, h, w, o), device=dev)
    launch("mb_launch_conv2d_nhwc_f32", ptr(d_x), ptr(d_w), ptr(d_y), n, h, w, c, o, 3, 3, 1, 1, None)
    want = x[..., 1].numpy().astype(np.float64)[..., None] * wt[:, 1, 1, 1].numpy().astype(np.float64)
    # (a product below the smallest normal number is rounded to a multiple of 2^-149)
    assert np.all(np.abs(d_y.cpu().numpy() - want) <= 2.0 ** -22 * want + 2.0 ** -149)
