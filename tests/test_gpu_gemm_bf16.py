"""bf16 GEMM (fp32 accumulate, bf16 out) on the GPU vs the float64 oracle.

Gate (benchmark configuration): rtol 1e-2 against the fp32-accumulated product, atol 1e-4.
Stronger check: with fp32 accumulation the error before rounding is ~1e-6
relative, far below half a bf16 ulp, so wherever |C| is not tiny (above 1% of
its RMS, where a bf16 ulp still dwarfs the fp32 accumulation noise) the
kernel's output must be the round-to-nearest-even bf16 of the exact product
within one bf16 ulp, and equal to it for almost every element."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import BF16_TILE_SHAPES, assert_close, launch, ptr, run_registry, seeded
from metalbench_amd import native

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _check_rounding(got_bits, exact, what, min_equal=0.99):
    want_bits = oracle.f32_to_bf16_bits(exact.astype(np.float32))
    # ordered distance in bf16 ulps (sign-magnitude -> two's complement)
    def ordered(b):
        b = b.astype(np.int32)
        return np.where(b & 0x8000, -(b & 0x7FFF), b)
    ulps = np.abs(ordered(got_bits) - ordered(want_bits))
    ulps = ulps[np.abs(exact) >= 0.01 * np.sqrt(np.mean(exact * exact))]
    assert ulps.max() <= 1, f"{what}: max {ulps.max()} bf16 ulps off the rounded exact product"
    frac = float(np.mean(ulps == 0))
    assert frac >= min_equal, f"{what}: only {frac:.4f} of elements equal the rounded exact product"


@pytest.mark.parametrize("m,n,k", [
    (256, 256, 64), (512, 256, 128), (256, 512, 512), (300, 260, 72), (1, 8, 8), (17, 24, 40),
    (256, 256, 8), (513, 1000, 200), (5, 7, 3), (64, 300, 1000), (1024, 1024, 1024),
])
def test_matmul_bf16_shapes(mb, dev, m, n, k):
    a = seeded(m + 3 * k, (m, k), ("normal", 0.0, 0.02), "bf16")
    b = seeded(n + 5 * k, (k, n), ("normal", 0.0, 0.02), "bf16")
    d_a, d_b = a.to(dev), b.to(dev)
    d_c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    launch("mb_launch_matmul_bf16", ptr(d_a), ptr(d_b), ptr(d_c), m, n, k, None)
    exact = oracle.matmul(oracle.as_f64(a), oracle.as_f64(b))
    got = oracle.as_f64(d_c)
    assert_close(got, exact, 1e-2, 1e-4, f"matmul_bf16 {m}x{n}x{k}")
    _check_rounding(_bits(d_c), exact, f"matmul_bf16 {m}x{n}x{k}")


def _random_bf16_shapes(n, seed=71):
    """Seeded shapes: half ragged (guarded and element-wise kernels), half full
    256 x 256 tiles with K a multiple of 128 (the DMA kernel)."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        if i % 2:
            out.append((256 * int(rng.integers(1, 4)), 256 * int(rng.integers(1, 4)),
                        128 * int(rng.integers(1, 7))))
        else:
            out.append(tuple(int(v) for v in rng.integers(1, 700, size=3)))
    return out


@pytest.mark.parametrize("m,n,k", _random_bf16_shapes(8))
def test_matmul_bf16_random_shapes(mb, dev, m, n, k):
    test_matmul_bf16_shapes(mb, dev, m, n, k)


def test_matmul_bf16_identity_exact(mb, dev):
    a = seeded(11, (256, 512), ("normal", 0.0, 1.0), "bf16")
    eye = torch.eye(512, dtype=torch.bfloat16)
    d_a, d_e = a.to(dev), eye.to(dev)
    d_c = torch.zeros((256, 512), dtype=torch.bfloat16, device=dev)
    launch("mb_launch_matmul_bf16", ptr(d_a), ptr(d_e), ptr(d_c), 256, 512, 512, None)
    assert torch.equal(d_c.cpu(), a)


def test_large_mm_registry_config_full(mb):
    """The 8192^3 config: all 67,108,864 outputs against the float64 product
    of the same bf16 operands (a few seconds of float64 BLAS on the host), at
    the registry gate and to within one bf16 ulp of its rounding."""
    b, inputs, outs, _ = run_registry("large_mm", seed=0)
    A, B = inputs
    got = outs[0]
    assert tuple(got.shape) == (8192, 8192)
    exact = oracle.matmul(oracle.as_f64(A), oracle.as_f64(B))
    assert_close(oracle.as_f64(got), exact, b.rtol, b.atol, "large_mm")
    _check_rounding(_bits(got).ravel(), exact.ravel(), "large_mm")


def test_kernel_attrs_report_register_split(mb):
    """mb_kernel_attrs_get reports the ArchVGPR / AGPR / SGPR counts of the
    kernel's own code object: each wave of the bf16 GEMM keeps its 128 x 128
    accumulator tile, 8 x 8 16x16 MFMA tiles of 4 fp32 per lane (256 per lane),
    in AGPRs, so one wave per SIMD fits."""
    a = native.kernel_attrs(native.kernel_find("large_matmul_bf16"))
    assert a["agprs"] == 256 and 0 < a["arch_vgprs"] <= 256, a
    assert a["arch_vgprs"] + a["agprs"] <= 512 and a["sgprs"] > 0
    assert a["waves_per_simd"] == 1 and a["static_lds_bytes"] == 163840
    for name in native.kernel_names():
        attrs = native.kernel_attrs(native.kernel_find(name))
        assert attrs["arch_vgprs"] > 0 and 1 <= attrs["waves_per_simd"] <= 8, (name, attrs)


# Shapes away from full 256 x 256 tiles: ragged and odd sizes, one past and one short
# of a tile, of a 32-deep stage and of a chunk of 8, even and odd rows.  (Every tile by
# itself: test_matmul_bf16_every_tile.)
@pytest.mark.parametrize("m,n,k", [
    (3001, 3002, 136), (2815, 2900, 72), (3000, 3002, 70), (2049, 3970, 250),
    (1025, 2050, 322), (1000, 3000, 98), (1001, 3001, 97), (1023, 2047, 289),
    (513, 1026, 130), (511, 1023, 131),
    (33, 66, 34), (31, 65, 33), (130, 200, 1026), (129, 199, 1025),
    (17, 34, 2), (15, 33, 1), (16, 30, 4098), (17, 31, 4097),
])
@pytest.mark.parametrize("shift", [0, 1])
def test_matmul_bf16_tile_edges(mb, dev, m, n, k, shift):
    """Also with all three matrices 2 bytes off a 4-byte boundary (a C there is left to
    the kernel with 64-bit addresses); nothing is written around C, and an infinite row
    of A (whose values follow the row before it in memory) reaches only its own
    outputs."""
    a = seeded(m + k, (m, k), ("normal", 0.0, 1.0), "bf16")
    b = seeded(n + k, (k, n), ("normal", 0.0, 1.0), "bf16")
    bad = m // 2
    a[bad] = float("inf")
    buf = [torch.full((t.numel() + 16,), 7.0, dtype=torch.bfloat16, device=dev)
           for t in (a, b, torch.empty(m, n))]
    for d, t in zip(buf, (a, b)):
        d[shift:shift + t.numel()] = t.flatten().to(dev)
    launch("mb_launch_matmul_bf16", *[d.data_ptr() + 2 * shift for d in buf], m, n, k, None)
    c = buf[2].float().cpu().numpy()
    got = c[shift:shift + m * n].reshape(m, n).astype(np.float64)
    rows = np.arange(m) != bad
    A, B = oracle.as_f64(a)[rows], oracle.as_f64(b)
    # bf16 rounding (2^-8 of the result) and fp32 sums (2^-20 of the products' magnitudes)
    want = A @ B
    assert np.all(np.abs(got[rows] - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -20 * (np.abs(A) @ np.abs(B)))
    assert not np.isfinite(got[bad]).any() or k == 0
    assert np.all(c[:shift] == 7.0) and np.all(c[shift + m * n:] == 7.0)


def test_matmul_bf16_operand_past_2gb(mb, dev):
    """32-bit buffer offsets do not reach it: the kernels with 64-bit addresses."""
    for k in (72, 67):
        m, n = (2 ** 31) // (2 * k) + 300, 8
        gen = torch.Generator(device=dev).manual_seed(4)
        a = torch.empty((m, k), device=dev).uniform_(-1, 1, generator=gen).to(torch.bfloat16)
        b = torch.empty((k, n), device=dev).uniform_(-1, 1, generator=gen).to(torch.bfloat16)
        c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
        launch("mb_launch_matmul_bf16", ptr(a), ptr(b), ptr(c), m, n, k, None)
        rows = torch.tensor([0, 255, 256, m // 2, m - 257, m - 1], device=dev)
        want = oracle.matmul(oracle.as_f64(a[rows]), oracle.as_f64(b))
        assert_close(oracle.as_f64(c[rows]), want, 1e-2, 1e-3, f"past 2 GB, k {k}")
        assert torch.isfinite(c).all()


def test_matmul_bf16_very_wide_rows(mb, dev):
    """24 rows of this B are just over 2^32 bytes: k-rows past K must read as zero, not
    wrap around to B's start, where an infinity stands that column 100 does not have."""
    n, k = 89_500_000, 2
    at = (24 * n) % 2 ** 31 + 100       # what column 100 of row 24 would wrap to
    a = torch.ones((1, k), device=dev, dtype=torch.bfloat16)
    b = torch.ones((k, n), device=dev, dtype=torch.bfloat16)
    b[0, at] = float("inf")
    c = torch.zeros((1, n), device=dev, dtype=torch.bfloat16)
    launch("mb_launch_matmul_bf16", ptr(a), ptr(b), ptr(c), 1, n, k, None)
    assert torch.isinf(c[0, at])
    c[0, at] = 2.0
    assert (c == 2.0).all()


@pytest.mark.parametrize("m,n,k", [(2304, 2048, 128), (256, 512, 256)])
@pytest.mark.parametrize("shift", [1, 2, 4])
def test_matmul_bf16_full_tiles_into_unaligned_c(mb, dev, m, n, k, shift):
    """Full tiles, more and fewer than 64, with C off a 16-byte boundary."""
    a = seeded(m + k, (m, k), ("normal", 0.0, 1.0), "bf16").to(dev)
    b = seeded(n + k, (k, n), ("normal", 0.0, 1.0), "bf16").to(dev)
    buf = torch.full((m * n + 16,), 7.0, dtype=torch.bfloat16, device=dev)
    launch("mb_launch_matmul_bf16", ptr(a), ptr(b), buf.data_ptr() + 2 * shift, m, n, k, None)
    c = torch.full((m, n), 7.0, dtype=torch.bfloat16, device=dev)
    launch("mb_launch_matmul_bf16", ptr(a), ptr(b), ptr(c), m, n, k, None)
    got = buf.float().cpu().numpy()
    assert np.all(got[:shift] == 7.0) and np.all(got[shift + m * n:] == 7.0)
    A, B = oracle.as_f64(a), oracle.as_f64(b)
    want, size = A @ B, np.abs(A) @ np.abs(B)
    for x in (got[shift:shift + m * n].reshape(m, n), c.float().cpu().numpy()):
        assert np.all(np.abs(x - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -20 * size)


def test_matmul_bf16_more_rows_than_small_tiles_can_launch(mb, dev):
    """2^30 - 1 rows of one odd-shaped element: 2^24 tiles of 64 rows would be 2^32
    threads, one more than a launch may have."""
    m = 2 ** 30 - 1
    a = torch.arange(m, device=dev, dtype=torch.int32).remainder_(251).to(torch.bfloat16)
    b = torch.full((1,), 2.0, device=dev, dtype=torch.bfloat16)
    c = torch.zeros((m,), device=dev, dtype=torch.bfloat16)
    launch("mb_launch_matmul_bf16", ptr(a), ptr(b), ptr(c), m, 1, 1, None)
    for at in range(0, m, 2 ** 28):
        assert torch.equal(c[at:at + 2 ** 28], a[at:at + 2 ** 28] * 2.0)


@pytest.mark.parametrize("shape", [s for s, _, _ in BF16_TILE_SHAPES], ids=str)
@pytest.mark.parametrize("off", ["", "a", "b", "ab", "c"])
def test_matmul_bf16_every_tile(mb, dev, shape, off):
    """Every tile, for even and odd rows, with A, B or both 2 bytes off a 4-byte boundary
    (the tiles for odd rows then take even K and N as well) or C 4 bytes off a 16-byte
    one.  The infinite row and what surrounds C as in test_matmul_bf16_tile_edges."""
    m, n, k = shape
    gen = torch.Generator(device=dev).manual_seed(m + n + k)
    put = {"a": 0, "b": 0, "c": 2 if off == "c" else 0}
    put.update({x: 1 for x in off if x in "ab"})
    buf = {x: torch.full((r * c + 16,), 7.0, dtype=torch.bfloat16, device=dev)
           for x, r, c in (("a", m, k), ("b", k, n), ("c", m, n))}
    view = {x: buf[x][put[x]:put[x] + r * c].view(r, c) for x, r, c in (("a", m, k), ("b", k, n), ("c", m, n))}
    for x in "ab":
        view[x].copy_(torch.empty(view[x].shape, device=dev).normal_(generator=gen))
    bad = m // 2 if m > 1 else None
    if bad is not None:
        view["a"][bad] = float("inf")
    launch("mb_launch_matmul_bf16", *[view[x].data_ptr() for x in "abc"], m, n, k, None)
    rows = torch.ones(m, dtype=torch.bool, device=dev)
    if bad is not None:
        rows[bad] = False
        assert not torch.isfinite(view["c"][bad]).any()
    A, B = view["a"][rows].double(), view["b"].double()
    want = A @ B
    # bf16 rounding (2^-8 of the result) and fp32 sums (2^-20 of the products' magnitudes)
    assert ((view["c"][rows].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * (A.abs() @ B.abs())).all()
    assert (buf["c"][:put["c"]] == 7.0).all() and (buf["c"][put["c"] + m * n:] == 7.0).all()
