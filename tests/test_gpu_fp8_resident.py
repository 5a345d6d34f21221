"""Per-tensor FP8 calibrate + quantize in one kernel (csrc/quant.hip,
k_quant_resident) against the two-kernel path, bit for bit: QuantParams, e4m3
bytes, and the f16 decode through a reference-products linear.  Sizes at both
ends of the kernel's range (2^24 elements; 32 float4 per thread on every CU)
and just outside it; NaN, infinities, zeros; a barrier that gives up at once."""
import numpy as np
import pytest

from tokenvector.inference_amd import device as D

pytestmark = pytest.mark.gpu

LOW, HIGH = 2 ** 24, 8192 * 3072  # HIGH fills 256 CUs


@pytest.fixture(scope="module")
def ctx(hip):
    c = D.Context(0)
    yield c
    c.close()


def _x(n, case):
    r = np.random.default_rng(n % 1009)
    x = r.standard_normal(n, np.float32)
    x[r.integers(0, n, 999)] *= np.float32(30.0)
    if case == "nan_first":
        x[0] = np.nan
    elif case == "nan_inside":
        x[[7, n // 2, n - 1]] = np.nan
    elif case == "inf":
        x[[5, n - 2]] = np.inf, -np.inf
    elif case == "zeros":
        x[:] = 0.0
        x[3] = -0.0
    elif case == "subnormal_codes":
        x[0] = 3.0e4  # most codes are subnormal or zero
    return x


def _quant(ctx, dx, n, two_pass, spin=-1):
    dq = D.DeviceBuffer.from_host(ctx, np.full(n, 0xA5, np.uint8))
    p = D.params_buffer(ctx)
    ctx.set_tuning(D.TUNE_QUANT_TWO_PASS, 1 if two_pass else -1)
    ctx.set_tuning(D.TUNE_GRID_SPIN, spin)
    try:
        D.quantize_fp8_e4m3_dynamic_tensor(ctx, dx, n, dq, p)
        ctx.synchronize()
    finally:
        ctx.set_tuning(D.TUNE_QUANT_TWO_PASS, -1)
        ctx.set_tuning(D.TUNE_GRID_SPIN, -1)
    got = D.read_params(p), dq.download()
    dq.close()
    return got


@pytest.mark.parametrize("n,case", [
    (LOW - 4, "plain"), (LOW, "plain"), (LOW + 4, "plain"), (LOW + 2, "plain"),
    (HIGH - 4, "plain"), (HIGH, "plain"), (HIGH + 4, "plain"),
    (LOW, "nan_first"), (LOW + 4, "nan_inside"), (LOW, "inf"), (LOW, "zeros"),
    (LOW, "subnormal_codes")])
def test_fp8_single_pass(ctx, n, case):
    print(f"fp8 single pass n={n} {case}", flush=True)
    dx = D.DeviceBuffer.from_host(ctx, _x(n, case))
    want_p, want_q = _quant(ctx, dx, n, True)
    for spin in (-1, 0):
        p, q = _quant(ctx, dx, n, False, spin)
        for f in ("scale", "min_val", "max_val"):
            a, b = np.float32(getattr(p, f)), np.float32(getattr(want_p, f))
            assert a.tobytes() == b.tobytes(), (f, spin)
        assert np.array_equal(q, want_q), spin
    dx.close()


@pytest.mark.parametrize("case", ["plain", "inf"])
def test_fp8_single_pass_f16(ctx, case):
    """The f16 form, through QuantizedLinear with reference products."""
    m, n, k = 8192, 64, 2048  # m * k = 2^24
    print(f"fp8 single pass f16 {case}", flush=True)
    r = np.random.default_rng(3)
    w = (r.standard_normal((n, k)) * 0.02).astype(np.float32)
    dw = D.DeviceBuffer.from_host(ctx, w)
    db = D.DeviceBuffer.from_host(ctx, np.zeros(n, np.float32))
    dx = D.DeviceBuffer.from_host(ctx, _x(m * k, case))
    lin = D.QuantizedLinear.from_float(ctx, dw, n, k, db, D.WEIGHT_FP8)
    out = []
    for two_pass in (1, -1):
        dy = D.DeviceBuffer.from_host(ctx, np.full((m, n), 3, np.float32))
        ctx.set_tuning(D.TUNE_QUANT_TWO_PASS, two_pass)
        try:
            lin.forward(dx, m, dy, D.ACT_PER_TENSOR)
            ctx.synchronize()
        finally:
            ctx.set_tuning(D.TUNE_QUANT_TWO_PASS, -1)
        out.append(dy.download().view(np.uint32))
        dy.close()
    assert np.array_equal(out[0], out[1])
    for b in (dw, db, dx):
        b.close()
