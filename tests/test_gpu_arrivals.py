"""The arrival count that lets a kernel's last workgroup finish the call
(csrc/tkv_reduce.h, arrive_last): grids around its two forms (one word up to 64
workgroups, 16 groups above) and uneven groups, through calibrate_minmax (one
workgroup per 4096 elements, 512 at most) and the percentile's histogram
passes, called several times so that a count left behind shows."""
import numpy as np
import pytest

from tokenvector.inference_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [1, 2, 16, 63, 64, 65, 79, 80, 81, 255, 256, 257, 511, 512, 700])
def test_arrivals(hip, blocks):
    print(f"arrivals {blocks}", flush=True)
    ctx = D.Context(0)
    n = 4096 * blocks
    r = np.random.default_rng(blocks)
    for i in range(4):
        x = r.standard_normal(n, np.float32)
        x[r.integers(0, n)] = -9.0 - i
        dx, p = D.DeviceBuffer.from_host(ctx, x), D.params_buffer(ctx)
        D.calibrate_minmax(ctx, dx, n, 1, p)
        ctx.synchronize()
        assert D.read_params(p).max_val == 9.0 + i
        D.calibrate_percentile(ctx, dx, n, p, 50.0)
        ctx.synchronize()
        rank = int(min(n - 1, 0.5 * n))
        assert D.read_params(p).max_val == np.partition(np.abs(x), rank)[rank]
        dx.close()
    ctx.close()
