"""Channel profiles at the edges of their summation's split: x nodes about a
multiple of 64 (the nodes of one workgroup), rows fewer than its 16 waves, and
just past the 512 chunks, against the CPU restatement (oracle/diagnostics.py)
on the (random) state the solver returns.
Tolerance: both sides sum at most n = 528 FP64 terms in an order of their own,
so a mean is within n eps = 1.2e-13 of its terms' size: 1e-12 of the profile's
scale; a fluctuation's deviations are formed from two such means: 1e-11."""
import numpy as np
import pytest

import cudanavierstokes_amd as cns
from oracle import diagnostics as D
from tests.helpers import flush_print

pytestmark = pytest.mark.gpu

SIZES = [(64, 3, 3), (65, 4, 4), (63, 24, 22), (150, 23, 22)]


@pytest.mark.parametrize("mx,my,mz", SIZES, ids=["x".join(map(str, c)) for c in SIZES])
def test_profiles_at_split_edges(mx, my, mz):
    cfg = cns.channel(mx=mx, my=my, mz=mz, order=2, scheme="rk3", Ma=1.2, Re=2000.0, check_cfl=4)
    flush_print(f"[case] channel profiles {mx}x{my}x{mz}")
    with cns.Solver(cfg) as s:
        rng = np.random.default_rng(mx)
        shape = (mz, my, mx)
        s.set_state(rng.uniform(0.7, 1.3, shape), *(rng.uniform(-0.5, 1.0, shape) for _ in range(3)),
                    rng.uniform(9.0, 11.0, shape))
        state = s.get_state()
        prof = s.channel_profiles()
    for k, a in D.avg_chan(*state).items():
        scale = max(float(np.max(np.abs(a))), 1e-300)
        err = float(np.max(np.abs(prof[k] - a)))
        assert err <= (1e-11 if k.endswith("f") else 1e-12) * scale, (k, err, scale)
