"""FP64 classic RK4 with the accumulator formed in the third stage from the two
stage states before it: steps against the oracle's RK4, alone and in a batch,
for every stencil half width (the third stage runs the three-operand form of
the kernel), partial tiles, walls and general viscosity; relative L2 1e-12,
Linf 1e-10 as the other step tests."""
import numpy as np
import pytest

import cudanavierstokes_amd as cns
from tests.helpers import assert_close, flush_print, initial_fields, oracle_from, state_errors

pytestmark = pytest.mark.gpu

WALLS = dict(periodic_x=0, nonuniform_x=1, forcing=1, Lx=2.0, Ma=1.5, Re=3000.0, viscexp=0.7)
FLOWS = [
    ("box_o2", "random", dict(mx=18, my=17, mz=16, stencil_size=1, stencil_visc=1, Ma=0.4)),
    ("box_o4", "random", dict(mx=32, my=20, mz=11, stencil_size=2, stencil_visc=2, Ma=0.4)),
    ("box_o6", "random", dict(mx=16, my=33, mz=19, stencil_size=3, stencil_visc=2, Ma=0.4)),
    ("box_o8", "random", dict(mx=24, my=16, mz=40, stencil_size=4, stencil_visc=4, Ma=0.4)),
    ("walls_o6", "channel", dict(WALLS, mx=21, my=16, mz=24, stencil_size=3, stencil_visc=3)),
    ("walls_o8", "channel", dict(WALLS, mx=32, my=9, mz=17, stencil_size=4, stencil_visc=2)),
]


@pytest.mark.parametrize("name,kind,kw", FLOWS, ids=[f[0] for f in FLOWS])
def test_rk4_steps_alone_and_batched(name, kind, kw):
    cfg = cns.Config(scheme=2, check_cfl=2, check_bulk=2, **kw)
    flush_print(f"[case] rk4 accumulator {name} {cfg}")
    orc = oracle_from(cfg)
    f = initial_fields(kind, orc)
    orc.set_state(*f)
    orc.step(3)
    want = orc.get_state()
    with cns.Solver(cfg) as a, cns.Solver(cfg) as b:
        a.set_state(*f)
        a.step(3, outputs=False)
        assert_close(state_errors(a.get_state(), want), 1e-12, 1e-10, name)
        b.set_state(*f)
        with cns.Batch([b]) as batch:
            batch.step(3)
        assert_close(state_errors(b.get_state(), want), 1e-12, 1e-10, name + " batched")
        assert np.array_equal(a.scalars()["time"], b.scalars()["time"]) or np.isclose(a.scalars()["time"], b.scalars()["time"], rtol=1e-12)
