"""GPU parity of calibrate_mse's one-pass form (csrc/calib.hip: 16 .. 31
candidates from 2^21 elements on, 32 .. 39 from 2^18, 40 .. 64 from 2^17)
against the CPU oracle (engine.tkv:165-197).

The chosen threshold must be the oracle's: two candidates' errors differ by far
more than the rounding of either sum except where they tie exactly, and then
the inputs below have one candidate that is better than both.
"""
from fractions import Fraction

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


def _choose(ctx, x, nc, off=0):
    dx = D.DeviceBuffer.from_host(ctx, np.concatenate([np.zeros(off, np.float32), x]))
    p = D.params_buffer(ctx)
    out = []
    for _ in range(2):
        D.calibrate_mse(ctx, dx.ptr + 4 * off, x.size, p, nc)
        out.append(D.read_params(p))
    p.close()
    dx.close()
    assert _bits(out[0]) == _bits(out[1])
    return out[0]


def _bits(q):
    v = np.array([q.scale, q.min_val, q.max_val], np.float32)
    return (q.zero_point, *np.where(np.isnan(v), np.float32(np.nan), v).view(np.uint32).tolist())


def _x(n, seed, heavy=True):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(n).astype(np.float32)
    return O.add_outliers(x, 0.001, 3, 4, 20.0) if heavy else x


@pytest.mark.parametrize("n,nc", [(131071, 32), (131072, 31), (131072, 32), (131073, 50),
                                  (262147, 64), (262147, 65), (1048575, 31), (1048576, 16),
                                  (1048579, 31), (1048576, 15), (2100001, 17), (2100001, 64),
                                  (2097151, 16), (2097152, 16), (2097155, 31), (2097152, 15),
                                  (262143, 32), (262144, 32), (262145, 39),
                                  (131071, 40), (131072, 40)])
def test_sizes_and_candidates(ctx, n, nc):
    """Both sides of each line of the rule; n past whole float4 groups, and x one
    float past a 16-byte boundary."""
    print(f"n={n} nc={nc}", flush=True)
    x = _x(n, n + nc)
    assert _bits(_choose(ctx, x, nc)) == _bits(O.calibrate_mse(x, nc))
    y = _x(n, n - nc, heavy=False)
    assert _bits(_choose(ctx, y, nc, 1)) == _bits(O.calibrate_mse(y, nc))


def _special(n):
    base = _x(n, 9)
    first, inside, inf, big = (base.copy() for _ in range(4))
    first[0] = np.nan
    inside[n // 2] = np.nan
    inf[3] = -np.inf
    big[7] = np.float32(3.4e38)
    relu = np.maximum(base, 0)
    sub = (base * np.float32(1e-41)).astype(np.float32)
    eighths = np.round(_x(n, 10, heavy=False) * 8).astype(np.float32) / 8
    return {"nan-first": first, "nan-inside": inside, "inf": inf, "big": big, "relu": relu,
            "tiny": base * np.float32(1e-25), "subnormal": sub, "eighths": eighths,
            "zero": np.zeros(n, np.float32), "equal": np.full(n, -0.75, np.float32),
            "all-nan": np.full(n, np.nan, np.float32), "large": base * np.float32(1e36)}


@pytest.mark.parametrize("n", [150001])
def test_special_values(ctx, n):
    for name, x in _special(n).items():
        print(name, flush=True)
        assert _bits(_choose(ctx, x, 50)) == _bits(O.calibrate_mse(x, 50)), name


# Values and counts for which candidates 6 and 7 of 16 differ by 1.2e-13 of
# their error, 30 times what the f64 sums of the bins may be off by; offsets
# rounded to 2^-38 of a cell (a fixed point that has to hold the sum of 2^17
# elements of up to 2^7 cells) make it 9e-14 the other way round.
CLOSE = {31.90129852294922: 792368, 91.46357727050781: 63517, 247.45388793945312: 13182337,
         47.75067138671875: 15823224, 288.6236267089844: 3692984, 1000.0: 1, 8.333157539367676: 1}


def test_values_that_repeat(ctx):
    """2^25 elements of seven values, whose rounding does not average out: the
    candidate with the least error in exact arithmetic."""
    nc, am = 16, max(CLOSE)
    mse = []
    for c in range(1, nc + 1):
        step = Fraction(am) * c / nc / 127
        mse.append(sum(k * (Fraction(v) - min(round(Fraction(v) / step), 127) * step) ** 2
                       for v, k in CLOSE.items()))
    best = mse.index(min(mse)) + 1
    x = np.repeat(np.array(list(CLOSE), np.float32), list(CLOSE.values()))
    assert x.size == 2 ** 25
    x = np.ascontiguousarray(x.reshape(4096, -1).T).reshape(-1)
    print(f"n={x.size} nc={nc} best={best}", flush=True)
    assert _choose(ctx, x, nc).max_val == np.float32(am * best / nc)


# around and past the elements between two flushes of the bins to their f64 rows
# (28 float4 per thread of 256 x 1024), aligned and not
@pytest.mark.parametrize("n,off,clip", [(28 * 2 ** 20 - 4, 0, 0), (28 * 2 ** 20, 0, 0),
                                        (28 * 2 ** 20 + 4, 0, 0.5), (28 * 2 ** 20 + 5, 1, 0),
                                        (57 * 2 ** 20 + 3, 0, 0), (2 ** 21 + 7, 0, 1e-3)])
def test_flushes(ctx, n, off, clip):
    """Clipped: most elements in the last bin, which has a slot per lane."""
    print(f"n={n} off={off} clip={clip}", flush=True)
    x = _x(n, n % 1000003)
    if clip:
        x = np.clip(x, -np.float32(clip), np.float32(clip))
    assert _bits(_choose(ctx, x, 20, off)) == _bits(O.calibrate_mse(x, 20))
