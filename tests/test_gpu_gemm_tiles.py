"""The GEMM's automatic tile choice at sizes on both sides of its lines
(csrc/gemm_kernels.h, pick_cfg): 64x64 and 128x128 tiles with 256-byte K slices
(row strides that are a multiple of 256), 64x128 tiles of 8 waves, and the
tiles they leave the rest to.  INT8 sums and QLinearMatMul against exact
arithmetic; both FP8 forms bit-identical to the forced 64x128 configuration
(every configuration adds the K steps in the same order)."""
import numpy as np
import pytest

import oracle as O
from tokenvector.inference_amd import device as D

pytestmark = pytest.mark.gpu

# one tile, ragged tiles, 256 tiles of 64x64 exactly, K of one and three slices
# (64x64); K % 256 == 128 and more tiles than CUs (64x128); one and two rounds
# (128x128 from three slices on); K % 256 == 128 past them (64x128 of 4
# waves, warp-specialised); one round more with 128x128 tiles than with 128x192
# (warp-specialised)
SHAPES = [(33, 1, 256), (65, 129, 768), (1024, 1024, 256), (700, 1500, 384), (1100, 1900, 256),
          (1100, 1900, 768), (3001, 769, 256), (3001, 2304, 512), (3001, 2304, 768),
          (3001, 769, 384), (2050, 2304, 128), (4100, 2300, 768)]


@pytest.fixture(scope="module")
def ctx(hip):
    c = D.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_automatic_tiles(ctx, m, n, k):
    print(f"gemm tiles {m}x{n}x{k}", flush=True)
    r = np.random.default_rng(m + n + k)
    a = r.integers(-128, 128, (m, k)).astype(np.int8)
    w = r.integers(-128, 128, (n, k)).astype(np.int8)
    da, dw = D.DeviceBuffer.from_host(ctx, a), D.DeviceBuffer.from_host(ctx, w)
    dacc = D.DeviceBuffer.from_host(ctx, np.full((m, n), 3, np.int32))
    D.matmul_int8_accum(ctx, da, dw, m, n, k, dacc)
    acc = a.astype(np.float64) @ w.astype(np.float64).T  # exact
    assert np.array_equal(dacc.download().astype(np.float64), acc)

    sa, sw = np.float32(0.02), np.float32(0.003)
    sy = np.float32(np.sqrt(k) * 128 * 128 * sa * sw / 90.0)
    dq = D.DeviceBuffer.from_host(ctx, np.full((m, n), 3, np.int8))
    for zpa, zpw in ((-3, 5), (0, 0)):
        D.qlinear_matmul(ctx, da, sa, zpa, dw, sw, zpw, sy, 7, dq, m, n, k)
        s = (acc - zpw * a.astype(np.float64).sum(1)[:, None] - zpa * w.astype(np.float64).sum(1)[None, :]
             + float(k * zpa * zpw))
        want = np.clip(np.rint(s * (np.float64(sa) * np.float64(sw) / np.float64(sy))) + 7, -128, 127)
        assert np.array_equal(dq.download().astype(np.float64), want), (zpa, zpw)

    # finite e4m3 bytes
    ca = (a.view(np.uint8) & 0xF7).copy()
    cw = (w.view(np.uint8) & 0xF7).copy()
    fa, fw = D.DeviceBuffer.from_host(ctx, ca), D.DeviceBuffer.from_host(ctx, cw)
    dy = D.DeviceBuffer.from_host(ctx, np.zeros((m, n), np.float32))
    for fast in (False, True):
        D.matmul_fp8_e4m3(ctx, fa, fw, m, n, k, None, 0, None, None, dy, fast=fast)
        y = dy.download()
        ctx.set_tuning(D.TUNE_GEMM_CFG, 0)
        try:
            D.matmul_fp8_e4m3(ctx, fa, fw, m, n, k, None, 0, None, None, dy, fast=fast)
        finally:
            ctx.set_tuning(D.TUNE_GEMM_CFG, -1)
        assert np.array_equal(y.view(np.uint32), dy.download().view(np.uint32)), fast
    if m <= 65:
        want = O.matmul_fp8_e4m3(ca.astype(np.int32).reshape(-1) - 128,
                                 cw.astype(np.int32).reshape(-1) - 128, None, m, n, k)
        ctx.synchronize()
        D.matmul_fp8_e4m3(ctx, fa, fw, m, n, k, None, 0, None, None, dy)
        mag = np.abs(want).max()
        assert np.allclose(dy.download().reshape(-1), want, rtol=1e-5, atol=1e-5 * mag)
    for b in (da, dw, dacc, dq, fa, fw, dy):
        b.close()
