"""The attention output's consumer, o_proj: ehip_packed_gemm and
ehip_pack_weight_panels (kernels::PackedGemm / PackWeightPanels,
src/kernels/gemm.h:61-78) against the oracle's restatement of the reference's
scalar tile, which is bit-identical to the reference build.

Bars: the device pack is bit-exact; the GEMM meets the reference's own GEMM
tolerance (allclose rtol 1e-4, atol 1e-5 * sqrt(k), packed_gemm_test.cpp:180-184)
over its shape list and the benchmark configurations' o_proj shapes; repeated
calls are bit-identical (split-k partials added in split order)."""
from types import SimpleNamespace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# The reference's PackedGemm shapes (tests/unit/packed_gemm_test.cpp:132-145)
# and the configs' o_proj: C4 decode (256 rows, 4096 -> 4096), C2 decode
# (32 rows, 896 -> 896), a C3-sized chunk slice (600 rows).
SHAPES = [(16, 64, 64), (16, 64, 96), (16, 176, 64), (8, 64, 512), (1, 64, 64),
          (1, 2048, 512), (4, 2048, 8192), (33, 8192, 256), (130, 300, 70), (7, 1, 33),
          (65, 129, 1000), (5, 40, 17), (32, 896, 896)]
# The largest shapes run for the bf16 checkpoints the configs use (the CPU
# oracle's fp32 and fp16 passes at these sizes would dominate the suite).
CASES = ([(s, d) for s in SHAPES for d in ("bf16", "f16", "f32")] +
         [((256, 4096, 4096), "bf16"), ((600, 4096, 1024), "bf16")])


def _weights(orc, ehip_mod, n, k, dtype, seed):
    wf = orc.fill_normal(n * k, 0.0, 1.0, seed).reshape(n, k)
    if dtype == ehip_mod.WEIGHT_F32:
        return wf
    if dtype == ehip_mod.WEIGHT_BF16:
        return orc.to_bf16_bits(wf)
    return wf.astype(np.float16).view(np.uint16)


def _run(gctx, ehip_mod, x, w, dtype, bias):
    m, k = x.shape
    n = w.shape[0]
    dw = gctx.to_device(w)
    dwp = gctx.alloc(((n + 15) // 16) * k * 16 * w.itemsize)
    assert gctx.pack_weight_panels(dw, dtype, n, k, dwp) == 0, gctx.last_error()
    dx = gctx.to_device(x)
    db = gctx.to_device(bias) if bias is not None else None
    dy = gctx.alloc(m * n * 4)
    assert gctx.packed_gemm(dx, m, k, dwp, dtype, n, db, dy) == 0, gctx.last_error()
    gctx.sync()
    y = dy.download(np.float32, (m, n))
    wp = dwp.download(w.dtype, ((n + 15) // 16, k, 16))
    for b in (dw, dx, dy, db):
        if b is not None:
            b.free()
    return y, wp, dwp


@pytest.mark.parametrize("shape,dtype", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_packed_gemm_matches_reference_tile(gctx, ehip_mod, orc, shape, dtype):
    m, k, n = shape
    dt = {"bf16": ehip_mod.WEIGHT_BF16, "f16": ehip_mod.WEIGHT_F16, "f32": ehip_mod.WEIGHT_F32}[dtype]
    seed = 100 + m + k + n
    x = orc.fill_normal(m * k, 0.0, 1.0, seed).reshape(m, k)
    w = _weights(orc, ehip_mod, n, k, dt, seed + 1)
    bias = orc.fill_normal(n, 0.0, 1.0, seed + 2) if (m + n) % 2 else None
    print(f"[gemm] m={m} k={k} n={n} {dtype} bias={bias is not None}", flush=True)
    y, wp, dwp = _run(gctx, ehip_mod, x, w, dt, bias)
    dwp.free()
    want_wp = orc.pack_weight_panels(w)
    assert np.array_equal(wp.view(np.uint8), want_wp.view(np.uint8)), "device pack differs"
    ref = orc.packed_gemm(x, want_wp, dt, n, bias)
    atol = 1e-5 * np.sqrt(k)
    err = np.abs(y.astype(np.float64) - ref)
    bad = err > atol + 1e-4 * np.abs(ref)
    assert not bad.any(), (int(bad.sum()), float(err.max()))


def test_packed_gemm_split_k_is_deterministic(gctx, ehip_mod, orc):
    """The decode-shaped o_proj (256 rows) splits k over workgroups: two calls
    give the same bits, and match the oracle."""
    m, k, n = 256, 4096, 4096
    x = orc.fill_normal(m * k, 0.0, 1.0, 5).reshape(m, k)
    w = _weights(orc, ehip_mod, n, k, ehip_mod.WEIGHT_BF16, 6)
    dw, dx = gctx.to_device(w), gctx.to_device(x)
    dwp = gctx.alloc(n * k * 2)
    assert gctx.pack_weight_panels(dw, ehip_mod.WEIGHT_BF16, n, k, dwp) == 0
    outs = []
    for _ in range(2):
        dy = gctx.alloc(m * n * 4)
        assert gctx.packed_gemm(dx, m, k, dwp, ehip_mod.WEIGHT_BF16, n, None, dy) == 0
        gctx.sync()
        outs.append(dy.download(np.float32, (m, n)))
        dy.free()
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    for b in (dw, dx, dwp):
        b.free()


@pytest.mark.parametrize("m,k,n", [
    (1, 32, 16), (16, 96, 250), (17, 64, 256), (31, 128, 257), (33, 4096, 1111), (64, 160, 896),
    (65, 896, 896), (127, 64, 4112), (128, 544, 272), (129, 256, 512), (257, 2048, 1000),
    (2100, 64, 4096), (2100, 256, 4096), (300, 224, 512), (256, 224, 512), (257, 256, 250)])
def test_wide_tiles_at_their_edges(gctx, ehip_mod, orc, m, k, n):
    """bf16 weights with k % 32 == 0 (tiles of 16-128 rows x 256 columns): row
    and column remainders, odd step counts, k splits of the last round's tiles
    (2100 rows have one whole round of them), both sides of the line where short
    sums of many rows leave them (k < 256, m > 256), and x and y 4 bytes off a
    16-byte boundary. Bars, against 64 bits: the reference's GEMM tolerance, and
    1e-6 in the 2-norm, what fp32 sums of up to 4096 terms in groups give
    (6.5e-7 there; x in two planes: about 1.5e-6)."""
    x = orc.fill_normal(m * k, 0.0, 1.0, m + k).reshape(m, k)
    w = _weights(orc, ehip_mod, n, k, ehip_mod.WEIGHT_BF16, n + k)
    bias = orc.fill_normal(n, 0.0, 1.0, 9)
    dw, db = gctx.to_device(w), gctx.to_device(bias)
    dwp = gctx.alloc(((n + 15) // 16) * k * 32)
    assert gctx.pack_weight_panels(dw, ehip_mod.WEIGHT_BF16, n, k, dwp) == 0
    raw = np.zeros(m * k + 1, np.float32)
    raw[1:] = x.ravel()
    dx, dy = gctx.to_device(raw), gctx.alloc(4 * (m * n + 2))
    dy.upload(np.full(m * n + 2, 7.0, np.float32))
    off = [SimpleNamespace(ptr=b.ptr + 4) for b in (dx, dy)]
    assert gctx.packed_gemm(off[0], m, k, dwp, ehip_mod.WEIGHT_BF16, n, db, off[1]) == 0
    gctx.sync()
    out = dy.download(np.float32, (m * n + 2,))
    assert out[0] == 7.0 and out[-1] == 7.0, "wrote outside y"
    ref = x.astype(np.float64) @ orc.bf16_bits_to_f32(w).astype(np.float64).T + bias
    err = np.abs(out[1:-1].reshape(m, n) - ref)
    bad = err > 1e-5 * np.sqrt(k) + 1e-4 * np.abs(ref)
    assert not bad.any(), (int(bad.sum()), float(err.max()))
    assert np.linalg.norm(err) <= 1e-6 * np.linalg.norm(ref)
    for b in (dw, db, dwp, dx, dy):
        b.free()


@pytest.mark.parametrize("m,k,n", [(16, 64, 256), (32, 896, 896), (130, 4096, 512),
                                   (2100, 64, 4096)])
@pytest.mark.parametrize("wt", ["WEIGHT_BF16", "WEIGHT_F16", "WEIGHT_F32"])
def test_third_plane_of_x_reaches_y(gctx, ehip_mod, orc, wt, m, k, n):
    """x = 1 + 1.5 * 2^-9 + b * 2^-18 with b in -1, 0, 1: its bf16 planes are 1,
    1.5 * 2^-9 and b * 2^-18. Weights come in pairs (w, -w), w = +-1, so that
    y = 2^-18 sum(b w): only the third plane is left. Every partial sum of a
    step is exact in fp32 (from 2^5 down to 2^-18), so y is to a quarter unit."""
    rng = np.random.default_rng(m + k)
    b = rng.integers(-1, 2, (m, k))
    x = (1 + 1.5 * 2.0**-9 + b * 2.0**-18).astype(np.float32)
    assert np.array_equal(x.astype(np.float64), 1 + 1.5 * 2.0**-9 + b * 2.0**-18)
    w = np.repeat(rng.choice([-1, 1], (n, k // 2)), 2, axis=1)
    w[:, 1::2] *= -1
    dtype = getattr(ehip_mod, wt)
    raw = {"WEIGHT_F32": w.astype(np.float32), "WEIGHT_F16": w.astype(np.float16).view(np.uint16),
           "WEIGHT_BF16": (w.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)}[wt]
    dx, dw = gctx.to_device(x), gctx.to_device(raw)
    dwp, dy = gctx.alloc(((n + 15) // 16) * k * 16 * raw.itemsize), gctx.alloc(4 * m * n)
    assert gctx.pack_weight_panels(dw, dtype, n, k, dwp) == 0
    assert gctx.packed_gemm(dx, m, k, dwp, dtype, n, None, dy) == 0
    gctx.sync()
    got = dy.download(np.float32, (m, n)).astype(np.float64) * 2.0**18
    assert np.abs(got - b.astype(np.float64) @ w.T.astype(np.float64)).max() <= 0.25
    for buf in (dx, dw, dwp, dy):
        buf.free()


def test_packed_gemm_validates(gctx, ehip_mod):
    buf = gctx.alloc(4096)
    L_ = ehip_mod.lib()
    assert L_.ehip_packed_gemm(gctx.h, buf.ptr, 0, 4, buf.ptr, 1, 4, None, buf.ptr) == \
        ehip_mod.INVALID_ARGUMENT
    assert L_.ehip_packed_gemm(gctx.h, buf.ptr, 2, 4, buf.ptr, 7, 4, None, buf.ptr) == \
        ehip_mod.INVALID_ARGUMENT
    assert L_.ehip_packed_gemm(gctx.h, buf.ptr, 2, 4, buf.ptr + 2, 1, 4, None, buf.ptr) == \
        ehip_mod.INVALID_ARGUMENT
    assert L_.ehip_pack_weight_panels(gctx.h, buf.ptr, 1, 0, 4, buf.ptr) == \
        ehip_mod.INVALID_ARGUMENT
    buf.free()
