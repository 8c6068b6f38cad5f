"""Decoder sub-ops and adjacent GEMMs on the GPU vs the float64 oracle.

Each registry entry runs at the reference's own shape and tolerance (the
registry's rtol/atol), then at ragged shapes that take the kernels' scalar
and multi-block paths.  Inputs are seeded normal(0, 1), like the reference's;
for the attention blocks at ragged shapes the weights are scaled by 1/sqrt(D)
so that the softmax is not one-hot (a near-tie between two keys would then
decide the output)."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import assert_close, run_bound, run_registry, seeded

pytestmark = pytest.mark.gpu

f64 = oracle.as_f64


def _registry_check(name, want_fn):
    b, inputs, outs, _ = run_registry(name, seed=0, warmup=1, iters=2)
    want = want_fn(*[f64(t) for t in inputs])
    assert_close(f64(outs[0]), want, b.rtol, b.atol, name)


def test_rms_norm_registry():
    _registry_check("rms_norm", lambda x: oracle.rms_norm(x, 1e-5))


def test_fused_add_rms_norm_registry():
    _registry_check("fused_add_rms_norm", lambda x, r: oracle.fused_add_rms_norm(x, r, 1e-5))


def test_rms_norm_linear_registry():
    _registry_check("rms_norm_linear", lambda x, w: oracle.rms_norm_linear(x, w, 1e-5))


def test_rope_embedding_registry():
    _registry_check("rope_embedding", lambda x: oracle.rope_embedding(x, 10000.0))


def test_swiglu_registry():
    _registry_check("swiglu", oracle.swiglu)


def test_fused_qkv_projection_registry():
    _registry_check("fused_qkv_projection", oracle.matmul)


def test_matvec_registry():
    _registry_check("matvec", oracle.matmul)


def test_batch_mm_registry():
    _registry_check("batch_mm", oracle.matmul)


def test_llama_attention_registry():
    _registry_check("llama_attention", lambda x, wq, wo: oracle.llama_attention(
        x, wq, wo, n_heads=4, n_kv_heads=2, base=10000.0))


def test_llama_decoder_layer_registry():
    _registry_check("llama_decoder_layer", lambda x, wq, wo, wgu, wd: oracle.llama_decoder_layer(
        x, wq, wo, wgu, wd, n_heads=4, n_kv_heads=2, base=10000.0, eps=1e-5))


# ---- ragged shapes ------------------------------------------------------------------------

@pytest.mark.parametrize("rows,cols", [(7, 100), (33, 1000), (5, 4096), (1, 4)])
def test_rms_norm_shapes(mb, rows, cols):
    x = seeded(1, (rows, cols))
    (y,) = run_bound("rms_norm_f32", [(0, x)], [(1, (rows, cols))],
                     [(2, "u32", cols), (3, "f32", 1e-5)])
    assert_close(f64(y), oracle.rms_norm(f64(x), 1e-5), 1e-3, 1e-3, f"rms_norm {rows}x{cols}")


@pytest.mark.parametrize("rows,cols", [(33, 260), (3, 7)])
def test_fused_add_rms_norm_shapes(mb, rows, cols):
    x, r = seeded(2, (rows, cols)), seeded(3, (rows, cols))
    (y,) = run_bound("fused_add_rms_norm_f32", [(0, x), (1, r)], [(2, (rows, cols))],
                     [(3, "u32", cols), (4, "f32", 1e-5)])
    assert_close(f64(y), oracle.fused_add_rms_norm(f64(x), f64(r), 1e-5), 1e-3, 1e-3,
                 f"fused_add_rms_norm {rows}x{cols}")


# edges of the float4 counts that hold a row in registers, and the loop beyond 8192; the
# sum of up to 8196 squares in fp32, at least 64 adders wide, is within 140 ulp
@pytest.mark.parametrize("rows,cols", [(5, 4), (5, 256), (6, 260), (3, 512), (7, 516), (9, 1024), (2, 1028),
                                       (3, 2048), (1, 2052), (5, 4096), (2, 4100), (3, 8192), (2, 8196),
                                       (2, 1027)])
@pytest.mark.parametrize("add", [False, True])
def test_rms_norm_row_widths(mb, rows, cols, add):
    x, r = seeded(21, (rows, cols)), seeded(22, (rows, cols))
    name = "fused_add_rms_norm_f32" if add else "rms_norm_f32"
    n = 2 if add else 1
    (y,) = run_bound(name, [(0, x), (1, r)][:n], [(n, (rows, cols))], [(n + 1, "u32", cols), (n + 2, "f32", 1e-5)])
    want = oracle.fused_add_rms_norm(f64(x), f64(r), 1e-5) if add else oracle.rms_norm(f64(x), 1e-5)
    assert_close(f64(y), want, 2e-5, 2e-5, f"{name} {rows}x{cols}")


@pytest.mark.parametrize("m,n,k", [(70, 90, 130), (64, 64, 64), (1, 3, 5),
                                   # full 64 x 64 tiles: the small-problem kernel (K = 512),
                                   # then bf16 term products
                                   (128, 192, 512), (64, 320, 768), (192, 64, 1024)])
def test_rms_norm_linear_shapes(mb, m, n, k):
    x, w = seeded(4, (m, k)), seeded(5, (n, k))
    (y,) = run_bound("rms_norm_linear_f32", [(0, x), (1, w)], [(2, (m, n))],
                     [(3, "u32", m), (4, "u32", n), (5, "u32", k), (6, "f32", 1e-5)])
    assert_close(f64(y), oracle.rms_norm_linear(f64(x), f64(w), 1e-5), 1e-3, 1e-3,
                 f"rms_norm_linear {m,n,k}")


@pytest.mark.parametrize("m,n,k", [(100, 70, 36), (65, 130, 257)])
def test_swiglu_shapes(mb, m, n, k):
    x, wg, wu = seeded(6, (m, k)), seeded(7, (k, n)), seeded(8, (k, n))
    (y,) = run_bound("swiglu_f32", [(0, x), (1, wg), (2, wu)], [(3, (m, n))],
                     [(4, "u32", m), (5, "u32", n), (6, "u32", k)])
    assert_close(f64(y), oracle.swiglu(f64(x), f64(wg), f64(wu)), 1e-3, 1e-3, f"swiglu {m,n,k}")


@pytest.mark.parametrize("batch,m,n,k", [(3, 70, 50, 33), (2, 64, 128, 256), (2, 64, 128, 512)])
def test_batch_mm_shapes(mb, batch, m, n, k):
    a, b = seeded(9, (batch, m, k)), seeded(10, (batch, k, n))
    (c,) = run_bound("batch_matmul_f32", [(0, a), (1, b)], [(2, (batch, m, n))],
                     [(3, "u32", m), (4, "u32", n), (5, "u32", k)])
    assert_close(f64(c), oracle.matmul(f64(a), f64(b)), 1e-3, 1e-3, f"batch_mm {batch,m,n,k}")


@pytest.mark.parametrize("m,k", [(77, 1001), (3, 4096), (5, 1)])
def test_matvec_shapes(mb, m, k):
    a, v = seeded(11, (m, k)), seeded(12, (k,))
    (y,) = run_bound("matvec_f32", [(0, a), (1, v)], [(2, (m,))], [(3, "u32", k)])
    assert_close(f64(y), oracle.matmul(f64(a), f64(v)), 1e-3, 1e-3, f"matvec {m,k}")


@pytest.mark.parametrize("s,d", [(5, 10), (300, 128), (1, 2)])
def test_rope_embedding_shapes(mb, s, d):
    x = seeded(13, (s, d))
    (y,) = run_bound("rope_embedding_f32", [(0, x)], [(1, (s, d))],
                     [(2, "u32", s), (3, "u32", d), (4, "f32", 10000.0)])
    assert_close(f64(y), oracle.rope_embedding(f64(x), 10000.0), 1e-4, 1e-5, f"rope {s}x{d}")


def _attn_inputs(s, d, h, hkv, seed):
    dh = d // h
    x = seeded(seed, (s, d))
    wq = seeded(seed + 1, (d, d + 2 * hkv * dh), ("normal", 0.0, d ** -0.5))
    wo = seeded(seed + 2, (d, d), ("normal", 0.0, d ** -0.5))
    return x, wq, wo


@pytest.mark.parametrize("s,d,h,hkv", [(70, 256, 4, 1), (1, 128, 4, 2), (130, 128, 1, 1),
                                       (64, 256, 8, 8)])
def test_llama_attention_shapes(mb, s, d, h, hkv):
    x, wq, wo = _attn_inputs(s, d, h, hkv, 20)
    (y,) = run_bound("llama_attention_f32", [(0, x), (1, wq), (2, wo)], [(3, (s, d))],
                     [(4, "u32", s), (5, "u32", d), (6, "u32", h), (7, "u32", hkv),
                      (8, "f32", 10000.0)])
    want = oracle.llama_attention(f64(x), f64(wq), f64(wo), n_heads=h, n_kv_heads=hkv)
    assert_close(f64(y), want, 1e-2, 1e-2, f"llama_attention {s,d,h,hkv}")


@pytest.mark.parametrize("s,d,h,hkv,ff", [(100, 256, 8, 2, 320), (1, 128, 4, 2, 256),
                                          (65, 128, 2, 1, 100)])
def test_llama_decoder_layer_shapes(mb, s, d, h, hkv, ff):
    x, wq, wo = _attn_inputs(s, d, h, hkv, 30)
    wgu = seeded(34, (d, 2 * ff), ("normal", 0.0, d ** -0.5))
    wd = seeded(35, (ff, d), ("normal", 0.0, ff ** -0.5))
    (y,) = run_bound("llama_decoder_layer_f32",
                     [(0, x), (1, wq), (2, wo), (3, wgu), (4, wd)], [(5, (s, d))],
                     [(6, "u32", s), (7, "u32", d), (8, "u32", h), (9, "u32", hkv),
                      (10, "u32", ff), (11, "f32", 10000.0), (12, "f32", 1e-5)])
    want = oracle.llama_decoder_layer(f64(x), f64(wq), f64(wo), f64(wgu), f64(wd), n_heads=h,
                                      n_kv_heads=hkv, base=10000.0, eps=1e-5)
    assert_close(f64(y), want, 1e-2, 1e-2, f"llama_decoder_layer {s,d,h,hkv,ff}")


def _attention_f32(x, wqkv, h, hkv):
    """Attention in float32 on the CPU (angles in float64), the heads side by side."""
    s, d = x.shape
    dh = d // h
    qkv = x @ wqkv
    ang = torch.arange(s, dtype=torch.float64)[:, None] * 10000.0 ** (-torch.arange(0, dh, 2) / dh)
    c, sn = torch.cos(ang).float(), torch.sin(ang).float()

    def rope(t):
        a, b = t[:, 0::2], t[:, 1::2]
        return torch.stack((a * c - b * sn, a * sn + b * c), dim=-1).reshape(s, dh)

    out = []
    for i in range(h):
        j = d + i // (h // hkv) * dh
        p = torch.softmax(rope(qkv[:, i * dh:(i + 1) * dh]) @ rope(qkv[:, j:j + dh]).T * dh ** -0.5, -1)
        out.append(p @ qkv[:, j + hkv * dh:j + (hkv + 1) * dh])
    return torch.cat(out, 1)


@pytest.mark.parametrize("s,d,h,hkv", [(1, 64, 2, 1), (15, 64, 1, 1), (17, 96, 3, 3),
                                       (33, 128, 4, 2), (64, 128, 1, 1), (65, 128, 1, 1),
                                       (256, 64, 2, 2), (127, 256, 2, 1), (129, 128, 1, 1),
                                       (257, 192, 3, 1), (530, 128, 4, 1)])
def test_attention_tile_edges(mb, s, d, h, hkv):
    """Partial tiles of queries and keys, waves without keys, each head size; W_o = 1, so
    the output is the attention itself."""
    x, wq, _ = _attn_inputs(s, d, h, hkv, 50)
    eye = torch.eye(d)
    want = oracle.llama_attention(f64(x), f64(wq), f64(eye), n_heads=h, n_kv_heads=hkv)
    (y,) = run_bound("llama_attention_f32", [(0, x), (1, wq), (2, eye)], [(3, (s, d))],
                     [(4, "u32", s), (5, "u32", d), (6, "u32", h), (7, "u32", hkv),
                      (8, "f32", 10000.0)])
    # fp32 throughout, in another order than the CPU's fp32 evaluation: its error, times four
    tol = 4 * np.abs(f64(_attention_f32(x, wq, h, hkv)) - want).max()
    assert np.abs(f64(y) - want).max() <= tol

    # The layer with W_down = 0 is x + attention(rmsnorm(x)), fp64 up to the attention's
    # output, which is then rounded, multiplied by W_o = 1 and added: four roundings at most.
    ff = 64
    (y,) = run_bound("llama_decoder_layer_f32",
                     [(0, x), (1, wq), (2, eye), (3, seeded(54, (d, 2 * ff))),
                      (4, torch.zeros(ff, d))], [(5, (s, d))],
                     [(6, "u32", s), (7, "u32", d), (8, "u32", h), (9, "u32", hkv),
                      (10, "u32", ff), (11, "f32", 10000.0), (12, "f32", 1e-5)])
    attn = oracle.llama_attention(oracle.rms_norm(f64(x), 1e-5), f64(wq), f64(eye), n_heads=h,
                                  n_kv_heads=hkv)
    assert (np.abs(f64(y) - (f64(x) + attn)) <= 2.0 ** -22 * (np.abs(f64(x)) + np.abs(attn))).all()


@pytest.mark.parametrize("dh", [32, 64, 128])
def test_attention_scores_are_summed_in_short_chains(mb, dh):
    """No further from 64 bits than q.k in four interleaved fp32 chains and p.v in one, in
    the mean over ten inputs.  q, k and v are columns of x (projections of ones and zeros,
    so exact); the tenth allowed above is for the spread of a mean over ten."""
    s, got_sq, chains_sq = 62, 0.0, 0.0
    eye = np.eye(dh, dtype=np.float32)
    w = torch.from_numpy(np.concatenate([eye, eye[:, ::-1], eye], 1).copy())
    ang = np.arange(s)[:, None] * 10000.0 ** (-np.arange(0, dh, 2) / dh)
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)

    def fma(a, b, c):
        return (a.astype(np.float64) * b + c).astype(np.float32)

    def rope(t):
        a, b = t[:, 0::2], t[:, 1::2]
        return np.stack((fma(a, cos, -(b * sin)), fma(a, sin, b * cos)), -1).reshape(s, dh)

    for seed in range(10):
        x = seeded(80 + seed, (s, dh))
        (y,) = run_bound("llama_attention_f32", [(0, x), (1, w), (2, torch.from_numpy(eye))], [(3, (s, dh))],
                         [(4, "u32", s), (5, "u32", dh), (6, "u32", 1), (7, "u32", 1), (8, "f32", 10000.0)])
        want = oracle.llama_attention(f64(x), f64(w), eye.astype(np.float64), n_heads=1, n_kv_heads=1)
        v = x.numpy()
        q, k = rope(v), rope(v[:, ::-1])
        part = [np.zeros((s, s), np.float32) for _ in range(4)]
        for d in range(dh):
            part[d % 4] = fma(q[:, d, None], k[None, :, d], part[d % 4])
        sc = ((part[0] + part[1]) + (part[2] + part[3])) * np.float32(dh ** -0.5)
        p = np.exp(sc - sc.max(1, keepdims=True))
        out = np.zeros((s, dh), np.float32)
        for j in range(s):
            out = fma(p[:, j, None], v[None, j], out)
        out /= p.sum(1, keepdims=True, dtype=np.float32)
        got_sq += ((f64(y) - want) ** 2).sum()
        chains_sq += ((out - want) ** 2).sum()
    ratio = (got_sq / chains_sq) ** 0.5
    print("error over that of the chains: %.3f" % ratio, flush=True)
    assert ratio <= 1.1


def test_rejects_bad_shapes(mb):
    import ctypes  # noqa: F401
    from metalbench_amd import native
    x = seeded(40, (4, 96))
    with pytest.raises(native.NativeError):   # head dim 96 / 4 = 24: unsupported
        run_bound("llama_attention_f32", [(0, x), (1, seeded(41, (96, 96 + 2 * 24))),
                                          (2, seeded(42, (96, 96)))], [(3, (4, 96))],
                  [(4, "u32", 4), (5, "u32", 96), (6, "u32", 4), (7, "u32", 1),
                   (8, "f32", 10000.0)])
    with pytest.raises(native.NativeError):   # odd D
        run_bound("rope_embedding_f32", [(0, seeded(43, (3, 5)))], [(1, (3, 5))],
                  [(2, "u32", 3), (3, "u32", 5), (4, "f32", 10000.0)])


def _silu(v):
    return v / (1 + np.exp(-v))


@pytest.mark.parametrize("scale", [1.0, 1e-36])
@pytest.mark.parametrize("m,n,k", [(70, 67, 129), (130, 64, 640)])
def test_fused_products_of_values_the_split_cannot_hold(mb, m, n, k, scale):
    """The row scale, residual and SwiGLU epilogues over bf16 term products: rows of
    elements of size `scale` and one ordinary value that meets zeros, and (scale 1)
    an infinite weight, whose tile is multiplied a second time.  Sums are within
    2^-21 of the products' magnitudes (2^-22 and the row scale's rounding)."""
    x = seeded(60, (m, k)) * scale
    x[:, 0] = 1.0
    wg, wu = seeded(61, (k, n)) / scale, seeded(62, (k, n)) / scale
    wg[0], wu[0] = 0.0, 0.0
    if scale == 1.0:
        wu[5, 3] = float("inf")
    X, G, U = f64(x), f64(wg), f64(wu)
    inf = np.isinf(U).any(0)
    Uf = np.where(np.isinf(U), 0, U)
    xn = oracle.rms_norm(X, 1e-5)

    def near(got, want, bound):
        assert np.array_equal(got[:, inf], want[:, inf])
        assert np.all((np.abs(got - want) <= bound)[:, ~inf])

    (y,) = run_bound("rms_norm_linear_f32", [(0, x), (1, wu.T.contiguous())], [(2, (m, n))],
                     [(3, "u32", m), (4, "u32", n), (5, "u32", k), (6, "f32", 1e-5)])
    with np.errstate(all="ignore"):
        near(f64(y), xn @ U, 2.0 ** -21 * (np.abs(xn) @ np.abs(Uf)))

    # SwiGLU: silu's slope is at most 1.1; its exponential and division round a few times
    (y,) = run_bound("swiglu_f32", [(0, x), (1, wg), (2, wu)], [(3, (m, n))],
                     [(4, "u32", m), (5, "u32", n), (6, "u32", k)])
    g, u = X @ G, X @ Uf
    size = 1.1 * (np.abs(X) @ np.abs(G)) * np.abs(u) + np.abs(_silu(g)) * (np.abs(X) @ np.abs(Uf))
    with np.errstate(all="ignore"):
        near(f64(y), _silu(g) * (X @ U), 2.0 ** -21 * size + 2.0 ** -20 * np.abs(_silu(g) * u))


@pytest.mark.parametrize("scale", [1.0, 1e-36])
def test_layer_products_of_values_the_split_cannot_hold(mb, scale):
    """The prefill layer with W_o = 0: x + act W_down, where W_down's elements are of
    size `scale` but for one row of ones that meets zero activations, and (scale 1)
    hold an infinity.  70 x 576 x 576, 70 x 644 x 576 and 70 x 576 x 644 products."""
    s, d, h, hkv, ff = 70, 576, 9, 3, 644
    x, wq, _ = _attn_inputs(s, d, h, hkv, 70)
    wgu, wd = seeded(73, (d, 2 * ff)) * d ** -0.5, seeded(74, (ff, d)) * scale
    wgu[:, ff:] /= scale
    wgu[:, ff], wd[0] = 0.0, 1.0
    if scale == 1.0:
        wd[5, 9] = float("inf")
    (y,) = run_bound("llama_decoder_layer_f32",
                     [(0, x), (1, wq), (2, torch.zeros(d, d)), (3, wgu), (4, wd)], [(5, (s, d))],
                     [(6, "u32", s), (7, "u32", d), (8, "u32", h), (9, "u32", hkv),
                      (10, "u32", ff), (11, "f32", 10000.0), (12, "f32", 1e-5)])
    X, G, D = f64(x), f64(wgu), f64(wd)
    inf = np.isinf(D).any(0)
    Df = np.where(np.isinf(D), 0, D)
    xn = oracle.rms_norm(X, 1e-5)
    g, u = xn @ G[:, :ff], xn @ G[:, ff:]
    act = _silu(g) * u
    size = np.abs(xn) @ np.abs(G)
    d_act = 2.0 ** -21 * (1.1 * size[:, :ff] * np.abs(u) + np.abs(_silu(g)) * size[:, ff:]) + 2.0 ** -20 * np.abs(act)
    want, got = X + act @ Df, f64(y)
    bound = d_act @ np.abs(Df) + 2.0 ** -22 * (np.abs(act) @ np.abs(Df)) + 2.0 ** -23 * np.abs(want)
    assert np.all((np.abs(got - want) <= bound)[:, ~inf])
    assert np.array_equal(got[:, inf], np.sign(act[:, 5:6]) * np.inf * np.ones((1, inf.sum())))
