"""FP32 storage read back as FP64 fields (cns_get_state): the device forms
r = (hi + lo) + rho0, u = (rho u) / r, ... in FP64, so the result equals the
same numpy expressions on the stored pairs bit for bit.  Sizes: the smallest
grid, and point counts that are odd (the copy goes in halves) or no multiple
of a workgroup."""
import numpy as np
import pytest

import cudanavierstokes_amd as cns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("comp", [1, 0], ids=["compensated", "plain"])
@pytest.mark.parametrize("scheme", ["rk3", "rk4"])
@pytest.mark.parametrize("size", [(2, 2, 2), (5, 7, 9), (33, 17, 11), (64, 32, 20)])
def test_read_back_is_the_stored_state(size, scheme, comp):
    mx, my, mz = size
    cfg = cns.taylor_green(n=mx, order=2, scheme=scheme, precision=1, compensated=comp).replace(my=my, mz=mz)
    rng = np.random.default_rng(mx * 100 + my)
    n = mx * my * mz
    r = rng.uniform(0.5, 1.5, n)
    u, v, w = (rng.uniform(-1.0, 1.0, n) for _ in range(3))
    e = rng.uniform(150.0, 200.0, n)
    # the offsets are the means, summed in storage order
    rho0, e0 = np.add.accumulate(r)[-1] / n, np.add.accumulate(e)[-1] / n
    stored = []
    for x in (r - rho0, u * r, v * r, w * r, e - e0):
        hi = x.astype(np.float32)
        lo = (x - hi.astype(np.float64)).astype(np.float32)
        stored.append(hi.astype(np.float64) + (lo.astype(np.float64) if comp else 0.0))
    want = [stored[0] + rho0]
    want += [m / want[0] for m in stored[1:4]] + [stored[4] + e0]
    with cns.Solver(cfg) as s:
        s.set_state(r, u, v, w, e)
        got = s.get_state()
    for k, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a.reshape(-1), b), (size, k, np.max(np.abs(a.reshape(-1) - b)))
