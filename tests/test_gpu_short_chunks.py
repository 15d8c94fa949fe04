"""Default z chunks of small grids: the launch rule gives chunks of one to a
few planes, down to a single plane, where a workgroup's first plane is also
its last.  One right-hand side and two steps against the oracle at the
tolerances of the parity tests (relative L2 1e-12, Linf 1e-10 FP64)."""
import numpy as np
import pytest

import cudanavierstokes_amd as cns
from tests import cases
from tests.helpers import assert_close, flush_print, initial_fields, oracle_from, state_errors

pytestmark = pytest.mark.gpu

CHANNEL = dict(periodic_x=0, nonuniform_x=1, forcing=1, Lx=2.0, Ly=4 * np.pi / 3, Lz=4 * np.pi, Re=3000.0, Pr=0.72,
               Ma=1.5, viscexp=0.7, check_cfl=1, check_bulk=1)
GRIDS = [
    ("one_plane_o8", "random", dict(mx=24, my=24, mz=24, stencil_size=4, stencil_visc=4, Ma=0.5, scheme=2)),
    ("one_plane_partial_tiles_o6", "random", dict(mx=17, my=19, mz=13, stencil_size=3, stencil_visc=2, Ma=0.5, scheme=1)),
    ("nz_at_its_minimum_o8", "random", dict(mx=33, my=9, mz=8, stencil_size=4, stencil_visc=3, Ma=0.5, scheme=0)),
    ("channel_two_planes_o4", "channel", dict(CHANNEL, mx=40, my=48, mz=63, stencil_size=2, stencil_visc=2, scheme=0)),
]


@pytest.mark.parametrize("name,kind,kw", GRIDS, ids=[g[0] for g in GRIDS])
def test_short_chunks_match_the_oracle(name, kind, kw):
    cfg = cns.Config(**kw)
    flush_print(f"[case] short chunks {name} {cfg}")
    orc = oracle_from(cfg)
    f = initial_fields(kind, orc)
    orc.set_state(*f)
    with cns.Solver(cfg) as s:
        s.set_state(*f)
        assert_close(cases.rel_errors(s.rhs(), orc.rhs()), 1e-12, 1e-10, name + " rhs")
        orc.step(2)
        s.step(2, outputs=False)
        assert_close(state_errors(s.get_state(), orc.get_state()), 1e-12, 1e-10, name + " state")
