"""permute_cols (csrc/int4.hip) on both sides of the rule that sends many
elements through LDS row by row: cols around 1024 (four rows per workgroup, one)
and 16384 (the widest row), rows around perm_rows_from and remainders of four;
entries outside [0, cols) gather 0.  Copies: bit-equal."""
import numpy as np
import pytest

from tokenvector.inference_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [
    (1, 3072), (3, 16384), (341, 3072), (342, 3072), (1025, 1024), (4099, 255), (1366, 768),
    (1024, 1025), (255, 4096), (257, 4096), (223, 8192), (225, 8192), (767, 16384), (769, 16384),
    (90, 16385)])
def test_permute_cols(hip, rows, cols):
    print(f"permute {rows}x{cols}", flush=True)
    r = np.random.default_rng(rows + cols)
    x = r.standard_normal((rows, cols), np.float32)
    perm = r.permutation(cols).astype(np.int64)
    bad = r.integers(0, cols, 3)
    perm[bad] = -1, cols, 2 ** 40
    ctx = D.Context(0)
    dx, dp = D.DeviceBuffer.from_host(ctx, x), D.DeviceBuffer.from_host(ctx, perm)
    dy = D.DeviceBuffer.from_host(ctx, np.full((rows, cols), 7, np.float32))
    D.permute_cols(ctx, dx, rows, cols, dp, 0, dy)
    ok = (perm >= 0) & (perm < cols)
    want = np.where(ok, x[:, np.where(ok, perm, 0)], np.float32(0))
    assert np.array_equal(dy.download().view(np.uint32), want.view(np.uint32))
    for b in (dx, dp, dy):
        b.close()
    ctx.close()
