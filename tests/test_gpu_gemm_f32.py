"""fp32 GEMM (matmul_f32, sqr_mm, rect_mm) on the GPU vs the float64 oracle.

Tolerance: rtol = atol = 1e-4 for the sqr_mm benchmark config, scaled with
sqrt(K) for the normal(0,1) shapes where |C| grows with K."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import assert_close, launch, ptr, run_bound, run_registry, seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (1, 64, 64), (64, 1, 64), (64, 64, 1), (64, 64, 64), (65, 33, 17),
    (128, 256, 64), (100, 300, 96), (257, 129, 200), (512, 512, 512), (31, 1000, 36),
    # fewer than 128 64x64 tiles and K <= 512 take the small-problem kernel
    # (32x32 tiles, K over up to 16 waves): K = 32 (one wave), 464 (15 waves,
    # the last one's slice half past K), ragged M and N
    (32, 96, 32), (96, 64, 464), (70, 130, 256),
    # full tiles and whole 16-deep units on the kernel of bf16 term products, as
    # every other shape: 8 and 12 units per wave
    (1024, 512, 512), (192, 128, 768),
])
def test_matmul_f32_shapes(mb, dev, m, n, k):
    a = seeded(m * 1000 + k, (m, k), ("uniform", -1.0, 1.0))
    b = seeded(n * 1000 + k + 1, (k, n), ("uniform", -1.0, 1.0))
    d_a, d_b = a.to(dev), b.to(dev)
    d_c = torch.full((m, n), float("nan"), device=dev)
    launch("mb_launch_matmul_f32", ptr(d_a), ptr(d_b), ptr(d_c), m, n, k, None)
    want = oracle.matmul(a.numpy(), b.numpy())
    assert_close(d_c.cpu().numpy(), want, 1e-4, 1e-4, f"matmul_f32 {m}x{n}x{k}")


def _random_f32_shapes(n, seed=72):
    """Seeded shapes: half ragged, half full 64 x 64 tiles with K a multiple of
    256 from 512 (bf16 term products from K = 768, the small-problem kernel at
    K = 512 when there are fewer than 128 tiles)."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        if i % 2:
            out.append((64 * int(rng.integers(1, 9)), 64 * int(rng.integers(1, 9)),
                        256 * int(rng.integers(2, 5))))
        else:
            out.append(tuple(int(v) for v in rng.integers(1, 600, size=3)))
    return out


@pytest.mark.parametrize("m,n,k", _random_f32_shapes(8))
def test_matmul_f32_random_shapes(mb, dev, m, n, k):
    test_matmul_f32_shapes(mb, dev, m, n, k)


def test_matmul_f32_k0_gives_zeros(mb, dev):
    d_c = torch.full((8, 8), 5.0, device=dev)
    d_a = torch.zeros(1, device=dev)
    launch("mb_launch_matmul_f32", ptr(d_a), ptr(d_a), ptr(d_c), 8, 8, 0, None)
    assert torch.all(d_c.cpu() == 0.0)


# small-problem kernel, then bf16 term products: ragged and full tiles
@pytest.mark.parametrize("n", [192, 1000, 1024])
def test_matmul_f32_identity_exact(mb, dev, n):
    a = seeded(3, (n, n))
    eye = torch.eye(n)
    d_a, d_eye = a.to(dev), eye.to(dev)     # keep both alive across the launch
    d_c = torch.zeros((n, n), device=dev)
    launch("mb_launch_matmul_f32", ptr(d_a), ptr(d_eye), ptr(d_c), n, n, n, None)
    assert torch.equal(d_c.cpu(), a)


@pytest.mark.parametrize("name", ["sqr_mm", "rect_mm"])
def test_matmul_registry_config(mb, name):
    b, inputs, outs, _ = run_registry(name, seed=0)
    want = oracle.matmul(inputs[0].numpy(), inputs[1].numpy())
    tol = 1e-4 if name == "sqr_mm" else 1e-3
    assert_close(outs[0].numpy(), want, tol, tol, name)


# The split kernel's edges (64 x 64 tiles, 16-deep k units dealt to 4 waves, two
# LDS slots per wave): one past and one short of a tile and of a unit, 1 to 8 units per
# wave.  (In so few tiles K up to 64 runs element-wise on fp32 MFMA: the first three;
# waves without a unit: test_matmul_f32_short_k.)
@pytest.mark.parametrize("m,n,k", [(65, 63, 15), (63, 65, 17), (64, 64, 48), (129, 66, 65),
                                   (66, 127, 129), (1, 2, 191), (130, 1, 257), (200, 333, 512)])
@pytest.mark.parametrize("shift", [0, 1])
def test_matmul_f32_split_edges(mb, dev, m, n, k, shift):
    """Also from pointers 4 bytes off a 16-byte boundary, and with nothing written past C.

    Each element within 2^-22 sum |a b|: the term products left out are under
    2^-26 of |a b| each, and the sums round to 2^-24 a few dozen times."""
    a, b = seeded(m + k, (m, k)), seeded(n + k, (k, n))
    buf = [torch.full((t.numel() + 8,), 7.0, device=dev) for t in (a, b, torch.empty(m, n))]
    for d, t in zip(buf, (a, b)):
        d[shift:shift + t.numel()] = t.flatten().to(dev)
    launch("mb_launch_matmul_f32", *[d.data_ptr() + 4 * shift for d in buf], m, n, k, None)
    c = buf[2].cpu().numpy()
    got = c[shift:shift + m * n].reshape(m, n)
    A, B = a.numpy().astype(np.float64), b.numpy().astype(np.float64)
    assert np.all(np.abs(got - A @ B) <= 2.0 ** -22 * (np.abs(A) @ np.abs(B)))
    assert np.all(c[:shift] == 7.0) and np.all(c[shift + m * n:] == 7.0)


# K up to 36 with at most 256 tiles, and up to 64 with 64, run element-wise on fp32
# MFMA, other short K on the split kernel: both sides of these lines, one past and one
# short of a unit
@pytest.mark.parametrize("m,n,k", [(1027, 1025, 1), (1090, 1030, 7), (1100, 1030, 15), (1026, 1100, 33),
                                   (1024, 1023, 32), (1024, 1023, 33), (1021, 1021, 36), (1021, 1021, 37), (513, 511, 64), (511, 513, 63),
                                   (509, 511, 65), (16321, 2, 18), (2, 16399, 31), (1, 1, 1)])
def test_matmul_f32_short_k(mb, dev, m, n, k):
    """Every product is added with a rounding of at most 2^-24 of a partial sum (on the
    split kernel less often, see above), and no partial sum is above sum |a b|."""
    a, b = seeded(m + k, (m, k)), seeded(n + k, (k, n))
    buf = torch.full((m * n + 8,), 7.0, device=dev)
    d_a, d_b = a.to(dev), b.to(dev)
    launch("mb_launch_matmul_f32", ptr(d_a), ptr(d_b), ptr(buf), m, n, k, None)
    c = buf.cpu().numpy()
    A, B = a.numpy().astype(np.float64), b.numpy().astype(np.float64)
    bound = max(2.0 ** -22, k * 2.0 ** -24) * (np.abs(A) @ np.abs(B))
    assert np.all(np.abs(c[:m * n].reshape(m, n) - A @ B) <= bound)
    assert np.all(c[m * n:] == 7.0)


@pytest.mark.parametrize("m,n,k", [(70, 67, 129), (128, 192, 640)])
def test_matmul_f32_values_the_split_cannot_hold(mb, dev, m, n, k):
    """Infinities, NaN, values that round to a bf16 infinity, and rows or columns
    near the smallest normal number give what fp32 products give."""
    a, b = seeded(1, (m, k)), seeded(2, (k, n))
    a[3, 5], a[10, 1], a[20, 2] = float("inf"), float("nan"), 3.4e38
    b[:, 7] *= 1e-30
    b[2, 9] = 0.0
    for x, y in ((a, b), (seeded(3, (m, k)) * 1e-36, seeded(4, (k, n)) * 1e30),
                 (seeded(5, (m, k)) * 1e30, seeded(6, (k, n)) * 1e-37)):
        d_x, d_y = x.to(dev), y.to(dev)
        d_c = torch.zeros((m, n), device=dev)
        launch("mb_launch_matmul_f32", ptr(d_x), ptr(d_y), ptr(d_c), m, n, k, None)
        X, Y = x.numpy().astype(np.float64), y.numpy().astype(np.float64)
        with np.errstate(all="ignore"):
            want = (X @ Y).astype(np.float32)
        got = d_c.cpu().numpy()
        # rows that hold the values above sum to inf or NaN in fp64 as well, but a
        # sum with 3.4e38 may overflow in fp32 on the way
        rows = np.arange(m) != 20
        assert np.array_equal(np.isnan(got[rows]), np.isnan(want[rows]))
        fin = np.isfinite(want) & rows[:, None]
        assert np.array_equal(got[rows][np.isinf(want[rows])], want[rows][np.isinf(want[rows])])
        Xf = np.where(np.isfinite(X), X, 0)
        assert np.all(np.abs(got[fin] - want[fin]) <= (2.0 ** -20 * (np.abs(Xf) @ np.abs(Y)))[fin])


def test_matmul_f32_operand_past_2gb(mb, dev):
    """32-bit buffer offsets do not reach it: the kernel with 64-bit addresses."""
    m, n, k = 2 ** 23 + 5, 3, 67
    gen = torch.Generator(device=dev).manual_seed(4)
    a = torch.empty((m, k), device=dev).uniform_(-1, 1, generator=gen)
    b = torch.empty((k, n), device=dev).uniform_(-1, 1, generator=gen)
    c = torch.full((m, n), float("nan"), device=dev)
    launch("mb_launch_matmul_f32", ptr(a), ptr(b), ptr(c), m, n, k, None)
    rows = torch.tensor([0, 1, 63, 64, 2 ** 22, m - 66, m - 2, m - 1], device=dev)
    want = oracle.matmul(a[rows].cpu().numpy(), b.cpu().numpy())
    assert_close(c[rows].cpu().numpy(), want, 1e-4, 1e-4, "past 2 GB")
    assert torch.isfinite(c).all()


# Elements far below the rest of their row or column, and alone in a product: every
# term of the split has to survive, whatever stands beside it.
@pytest.mark.parametrize("e", [-100, -110, -115, -120, -126, -130, -140, -149])
def test_matmul_f32_small_elements_keep_their_bits(mb, dev, e):
    """A = [1, 0 .., v], B = [0; ..; w]: the product v w alone, v from 2^e on and w = 2^100 (or the
    other way round).  Both are powers of two or 24-bit numbers, so fp32 products would
    be exact up to one rounding; a subnormal v has the bits fp32 holds."""
    v = np.float32(1.37 * 2.0 ** e)
    for n, k in ((1, 2), (65, 2), (1, 66), (2, 67), (65, 68)):   # (K = 2: fp32 MFMA)
        a = torch.zeros((1, k))
        a[0, 0], a[0, k - 1] = 1.0, float(v)
        b = torch.zeros((k, n))
        b[k - 1] = 2.0 ** 100
        want = float(v) * 2.0 ** 100
        for x, y in ((a, b), (b.T.contiguous(), a.T.contiguous())):
            d_x, d_y = x.to(dev), y.to(dev)
            m, nn = x.shape[0], y.shape[1]
            d_c = torch.zeros((m, nn), device=dev)
            launch("mb_launch_matmul_f32", ptr(d_x), ptr(d_y), ptr(d_c), m, nn, k, None)
            got = d_c.cpu().numpy().astype(np.float64)
            assert np.all(np.abs(got - want) <= 2.0 ** -23 * want), (n, got.ravel()[0] / want - 1)


@pytest.mark.parametrize("m,n,k", [(70, 67, 129), (128, 192, 640)])
@pytest.mark.parametrize("scale", [1e-30, 1e-35, 1e-37])
def test_matmul_f32_mixed_magnitudes(mb, dev, m, n, k, scale):
    """One ordinary value in every row, met by a zero; the others carry the sum."""
    a, b = seeded(7, (m, k)) * scale, seeded(8, (k, n)) * 1e30
    a[:, 0], b[0] = 1.0, 0.0
    for x, y in ((a, b), (b.T.contiguous(), a.T.contiguous())):
        mm, nn = x.shape[0], y.shape[1]
        d_x, d_y = x.to(dev), y.to(dev)
        d_c = torch.zeros((mm, nn), device=dev)
        launch("mb_launch_matmul_f32", ptr(d_x), ptr(d_y), ptr(d_c), mm, nn, k, None)
        X, Y = x.numpy().astype(np.float64), y.numpy().astype(np.float64)
        assert np.all(np.abs(d_c.cpu().numpy() - X @ Y) <= 2.0 ** -22 * (np.abs(X) @ np.abs(Y)))


@pytest.mark.parametrize("dual", [False, True])
def test_matmul_f32_very_wide_rows(mb, dev, dual):
    """15 rows of this B are just over 2^32 bytes: k-rows past K must read as zero, not
    wrap around to B's start, where an infinity stands that column 100 does not have."""
    n = 71_600_000
    at = (15 * n) % 2 ** 30 + 100       # what column 100 of row 15 would wrap to
    a = torch.full((1, 1), 2.0, device=dev)
    b = torch.ones((1, n), device=dev)
    b[0, at] = float("inf")
    c = torch.zeros((1, n), device=dev)
    if dual:                            # SwiGLU: silu(a b) (a b)
        binds = [mb.make_binding(i, mb.ROLE_INPUT if i < 3 else mb.ROLE_OUTPUT, "f32", t.data_ptr(), t.numel() * 4)
                 for i, t in enumerate((a, b, b, c))]
        binds += [mb.make_binding(4 + i, mb.ROLE_SCALAR, "u32", value=v) for i, v in enumerate((1, n, 1))]
        mb.run(mb.kernel_find("swiglu_f32"), binds, 0, 1)
    else:
        launch("mb_launch_matmul_f32", ptr(a), ptr(b), ptr(c), 1, n, 1, None)
    want = 4.0 / (1.0 + float(np.exp(-2.0))) if dual else 2.0
    assert torch.isinf(c[0, at])
    c[0, at] = want
    assert (c - want).abs().max().item() <= 1e-6 * want


# sqr_mm's kernel (fp32 MFMA fed by DMA: full tiles, K a multiple of 256 from 512): the
# shortest K that reaches it, two and more trips of its loop, one tile and many
@pytest.mark.parametrize("m,n,k", [(1024, 512, 512), (64, 64, 768), (192, 128, 1024), (576, 640, 1280)])
def test_sqr_mm_full_tiles(mb, m, n, k):
    a, b = seeded(m + k, (m, k)), seeded(n + k, (k, n))
    (c,) = run_bound("sqr_matmul_f32", [(0, a), (1, b)], [(2, (m, n))],
                     [(3, "u32", m), (4, "u32", n), (5, "u32", k)])
    A, B = a.numpy().astype(np.float64), b.numpy().astype(np.float64)
    # a chain of k / 2 roundings to 2^-24 of a partial sum per K half, random in sign
    assert np.all(np.abs(c.numpy() - A @ B) <= 2.0 ** -20 * (np.abs(A) @ np.abs(B)))


@pytest.mark.parametrize("m,n,k", [(40000, 16001, 130), (100, 6_000_000, 5), (70, 9_000_000, 4)])
def test_matmul_f32_output_past_2gb(mb, dev, m, n, k):
    """C past 2 GB from small operands; the last shape's rows pass what a tile's 32-bit
    offsets reach."""
    gen = torch.Generator(device=dev).manual_seed(5)
    a = torch.empty((m, k), device=dev).uniform_(-1, 1, generator=gen)
    b = torch.empty((k, n), device=dev).uniform_(-1, 1, generator=gen)
    buf = torch.full((m * n + 64,), 7.0, device=dev)
    launch("mb_launch_matmul_f32", ptr(a), ptr(b), ptr(buf), m, n, k, None)
    c = buf[:m * n].view(m, n)
    for rows in range(0, m, 4000):
        A, B = a[rows:rows + 4000].double(), b.double()
        for cols in range(0, n, 1_000_000):
            Bc = B[:, cols:cols + 1_000_000]
            off = (c[rows:rows + 4000, cols:cols + 1_000_000] - A @ Bc).abs()
            assert (off <= 2.0 ** -22 * (A.abs() @ Bc.abs())).all(), (rows, cols)
    assert (buf[m * n:] == 7.0).all()
