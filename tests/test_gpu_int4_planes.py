"""GPU parity of the digit-plane INT4 GEMM (csrc/int4_planes.hip: products of
at least 1.6e8 multiply-adds, or 2.6e8 / 3.5e8 with group sizes 64 / 32 and no
column permutation, more where the columns are few (csrc/int4.hip, planes_pay);
K % 128 == 0, group sizes 32, 64 and multiples of 128) against the CPU oracle.

Every sum inside a group is exact there, and each output sees at most 4
roundings per group and 128 k, so the bound of the f64 form holds as it is:
|y - y_ref| <= 2 K 2^-53 sum_k |a_k w_k| + ulp(y_ref), and bit equality where
every partial sum of the reference is exact.
"""
import numpy as np
import pytest

import oracle as O
from tokenvector.inference_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(hip):
    c = D.Context(0)
    yield c
    c.close()


def _run(ctx, a, pk, sc, b, perm, m, n, k, gs):
    bufs = [D.DeviceBuffer.from_host(ctx, x) for x in (a, pk.astype(np.uint8), sc)]
    db = D.DeviceBuffer.from_host(ctx, b) if b is not None else None
    dp = D.DeviceBuffer.from_host(ctx, perm) if perm is not None else None
    dy = D.DeviceBuffer.from_host(ctx, np.full(m * n, 7.0, np.float32))
    D.matmul_int4_grouped(ctx, *bufs, db, dp, dy, m, n, k, gs)
    y = dy.download()
    for x in bufs + [db, dp, dy]:
        if x is not None:
            x.close()
    return y


def _check(y, a, pk, sc, b, perm, m, n, k, gs):
    ref = O.matmul_int4_grouped(a, pk, b, m, n, k, gs, sc, perm=perm)
    ap = np.asarray(a, np.float64).reshape(m, k)
    if perm is not None:
        ap = ap[:, perm]
    wd = np.asarray(O.dequantize_int4_grouped(pk, n, k, gs, sc), np.float64).reshape(n, k)
    with np.errstate(all="ignore"):
        bound = 2 * k * 2.0 ** -53 * (np.abs(ap) @ np.abs(wd).T).reshape(-1) + np.spacing(np.abs(ref))
        err = np.abs(y.astype(np.float64) - ref)
    fine = np.isfinite(ref)
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    same = ~fine & ~np.isnan(ref)
    assert np.array_equal(y[same], ref[same])
    assert np.all(err[fine] <= bound[fine])
    return ref


def _weights(n, k, gs, seed):
    return O.quantize_int4_grouped(O.gi_noise(n * k, seed, 0.02), n, k, gs)


# Ragged rows and columns (one row past a unit, one column past a tile), one
# chunk of K, K splits (few tiles), group scales per 32, 64, 128 and 256, the
# act-order gather, no bias.
@pytest.mark.parametrize("m,n,k,gs,perm,bias", [
    (385, 3300, 128, 128, False, True), (65, 1025, 3072, 128, False, True),
    (64, 768, 4096, 256, True, False), (257, 1000, 768, 32, True, True),
    (689, 257, 1536, 64, False, False), (320, 770, 768, 64, True, True),
    (72, 2304, 2176, 32, False, True)])
def test_shapes(ctx, m, n, k, gs, perm, bias):
    print(f"int4 planes {m}x{n}x{k} gs={gs} perm={perm}", flush=True)
    a = O.gi_noise(m * k, 3 + m, 1.0)
    pk, sc = _weights(n, k, gs, 5 + n)
    b = O.gi_noise(n, 9, 0.01) if bias else None
    p = np.random.default_rng(k).permutation(k).astype(np.int64) if perm else None
    y = _run(ctx, a, pk, sc, b, p, m, n, k, gs)
    ref = _check(y, a, pk, sc, b, p, m, n, k, gs)
    assert np.mean(y == ref) > 0.999
    assert np.array_equal(y, _run(ctx, a, pk, sc, b, p, m, n, k, gs))


@pytest.mark.parametrize("n,perm", [(40, False), (130, False), (130, True)])
def test_row_panels(ctx, n, perm):
    """K = 16384: the planes of 2176 rows take two passes (40 columns are too few
    for the planes)."""
    m, k, gs = 2176, 16384, 128
    print(f"int4 planes {m}x{n}x{k} perm={perm}", flush=True)
    a = O.gi_noise(m * k, 1, 1.0)
    pk, sc = _weights(n, k, gs, 2)
    b = O.gi_noise(n, 9, 0.01)
    p = np.random.default_rng(n).permutation(k).astype(np.int64) if perm else None
    y = _run(ctx, a, pk, sc, b, p, m, n, k, gs).reshape(m, n)
    rows = np.r_[0:2, 2046:2050, 2174:2176]
    sub = np.ascontiguousarray(a.reshape(m, k)[rows]).reshape(-1)
    _check(y[rows].reshape(-1), sub, pk, sc, b, p, rows.size, n, k, gs)


@pytest.mark.parametrize("kind", ["digits", "wide", "zeros", "special", "tiny"])
def test_value_ranges(ctx, kind):
    """Chunks of every number of digit planes, and units that the planes do
    not hold exactly: their tiles take the f64 form."""
    m, n, k, gs = 200, 1030, 1024, 128
    print(f"int4 planes values {kind}", flush=True)
    r = np.random.default_rng(11)
    a = O.gi_noise(m * k, 21, 1.0).reshape(m, k).copy()
    if kind == "digits":  # 1 .. 4 pairs of planes, chunk by chunk: small integers up to 2^-30
        for g in range(k // 128):
            s = a[:, 128 * g:128 * g + 128]
            if g % 4 == 0:
                s[:] = r.integers(-15, 16, s.shape)
            elif g % 4 == 1:
                s[:] = r.integers(-4000, 4001, s.shape)
            else:
                s[3::7, ::5] *= np.float32(2.0 ** -24)
    elif kind == "wide":  # rows of very different size; one unit needs the f64 form
        a[::3] *= np.float32(2.0 ** -9)
        a[70] *= np.float32(2.0 ** -60)
    elif kind == "zeros":
        a[:, 128:384] = 0.0
        a[64:128] = 0.0
        a[10] = -0.0
    elif kind == "special":
        a[5, 100] = np.inf
        a[5, 900] = -np.inf
        a[130, 640] = np.nan
        a[131, 641] = -np.inf
    else:  # f32 subnormals next to the smallest normals, and their own unit
        a *= np.float32(1e-37)
        a[64:128] = r.integers(-3, 4, (64, k)).astype(np.float32) * np.float32(1e-45)
    a = np.ascontiguousarray(a.reshape(-1))
    pk, sc = _weights(n, k, gs, 31)
    b = None if kind == "tiny" else O.gi_noise(n, 9, 0.01)
    y = _run(ctx, a, pk, sc, b, None, m, n, k, gs)
    _check(y, a, pk, sc, b, None, m, n, k, gs)


# One chunk of K unsplit, K splits with group sizes 128, 64 and 32.
@pytest.mark.parametrize("m,n,k,gs", [(385, 3300, 128, 128), (200, 1030, 1024, 128),
                                      (260, 1030, 1024, 64), (72, 2304, 2176, 32)])
def test_scales_not_finite(ctx, m, n, k, gs):
    """0 * scale is NaN for a NaN or infinite scale: over an activation unit
    that is zero (rows 0 .. 63, the first 128 k), over code 8, and in sums of
    both signs; products of one sign give an infinity."""
    print(f"int4 planes scales {m}x{n}x{k} gs={gs}", flush=True)
    a = O.gi_noise(m * k, 41, 1.0).reshape(m, k).copy()
    a[:64, :128] = 0.0
    a[66] = np.abs(a[66]) + np.float32(0.5)
    a[67] = -a[66]
    pk, sc = (np.array(v) for v in _weights(n, k, gs, 43))
    pk, sc = pk.reshape(n, k // 2), sc.reshape(n, k // gs)
    last = k // gs - 1
    sc[0, 0] = np.nan
    sc[3, last] = np.inf
    sc[300, 0] = -np.inf
    sc[n - 1, last] = np.inf
    pk[n - 1] = 0xFF       # every code 7: infinities where the activations have one sign
    sc[700, 0] = np.inf
    pk[700] = 0x8F         # code 7 and code 0 in turn
    pk[301] = 0x88         # a zero column whose scale is finite stays zero
    a, pk, sc = (np.ascontiguousarray(v.reshape(-1)) for v in (a, pk, sc))
    b = O.gi_noise(n, 9, 0.01)
    y = _run(ctx, a, pk, sc, b, None, m, n, k, gs)
    ref = _check(y, a, pk, sc, b, None, m, n, k, gs).reshape(m, n)
    assert np.isnan(ref[0, 0]) and ref[66, n - 1] == np.inf and ref[67, n - 1] == -np.inf
    assert np.isfinite(ref[:, 301]).all()


# Unsplit with group sizes 128, 64 and 32 (ragged rows and columns, a bias), K
# splits with 128 and 32.
@pytest.mark.parametrize("m,n,k,gs", [(385, 3300, 128, 128), (1000, 1030, 384, 64),
                                      (1300, 1030, 384, 32), (200, 1030, 1024, 128),
                                      (72, 2304, 2176, 32)])
@pytest.mark.parametrize("kind", ["one", "some", "all", "special"])
def test_flagged_chunks(ctx, m, n, k, gs, kind):
    """Values that the planes do not hold in one chunk of K, in some, in all of
    them: those chunks go through the f64 MFMA, the others through the planes."""
    print(f"int4 planes flags {kind} {m}x{n}x{k} gs={gs}", flush=True)
    a = O.gi_noise(m * k, 51, 1.0).reshape(m, k).copy()
    small = np.float32(1.2345e-13)  # 43 orders below the maximum
    if kind == "one":
        a[m - 1, k - 1] = small
    elif kind == "some":
        a[5, 3] = small
        a[40, k - 100] = -small
        a[64:128, k // 2:] = 0.0
        a[m - 3, k // 3] = np.inf
    elif kind == "all":
        a[::32, ::64] = small
    else:
        a[5, 100] = np.inf
        a[5, k - 28] = -np.inf
        a[65, 17] = np.nan
        a[m - 1, k - 1] = -np.inf
    a = np.ascontiguousarray(a.reshape(-1))
    pk, sc = _weights(n, k, gs, 53)
    b = O.gi_noise(n, 9, 0.01)
    y = _run(ctx, a, pk, sc, b, None, m, n, k, gs)
    _check(y, a, pk, sc, b, None, m, n, k, gs)
    assert np.array_equal(y, _run(ctx, a, pk, sc, b, None, m, n, k, gs), equal_nan=True)


def test_exact_where_the_reference_is(ctx):
    """Dyadic activations, scales and biases: every partial sum of the
    reference is exact, so every output is its bit for bit."""
    for m, n, k, gs in ((260, 700, 1024, 128), (110, 1100, 3072, 32)):
        print(f"int4 planes dyadic {m}x{n}x{k}", flush=True)
        r = np.random.default_rng(m)
        a = (r.integers(-2048, 2048, m * k) / 64.0).astype(np.float32)
        pk = r.integers(0, 256, n * k // 2).astype(np.int32)
        sc = (2.0 ** -r.integers(1, 6, n * k // gs)).astype(np.float32)
        b = (r.integers(-8, 8, n) / 8.0).astype(np.float32)
        y = _run(ctx, a, pk, sc, b, None, m, n, k, gs)
        assert np.array_equal(y, O.matmul_int4_grouped(a, pk, b, m, n, k, gs, sc))


def test_capture_without_workspaces(hip):
    """A fresh context captures a product whose planes have no workspace yet:
    the graph holds the f64 kernels, as it always could, and replays them."""
    m, n, k, gs = 2048, 1040, 128, 128
    c = D.Context(0)
    a = O.gi_noise(m * k, 3, 1.0)
    pk, sc = _weights(n, k, gs, 5)
    da, dw, ds = (D.DeviceBuffer.from_host(c, x) for x in (a, pk.astype(np.uint8), sc))
    dy = D.DeviceBuffer.from_host(c, np.zeros(m * n, np.float32))
    with D.Graph(c) as g:
        D.matmul_int4_grouped(c, da, dw, ds, None, None, dy, m, n, k, gs)
    for _ in range(3):
        D.memset(c, dy, 0, dy.nbytes)
        g.launch()
        c.synchronize()
        y = dy.download()
        rows = np.array([0, 31, 1000, m - 1])
        sub = np.ascontiguousarray(a.reshape(m, k)[rows]).reshape(-1)
        _check(y.reshape(m, n)[rows].reshape(-1), sub, pk, sc, None, None, rows.size, n, k, gs)
        D.matmul_int4_grouped(c, da, dw, ds, None, None, dy, m, n, k, gs)  # eager: planes
        c.synchronize()
    g.close()
    c.close()
