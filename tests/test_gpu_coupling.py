"""The grid-atom force walk at the edges of its shapes: lanes per atom (8 on a
narrow coupling, 16 by tiles of bins on a wide one), atoms that leave a wave or
a tile partly empty, and pair counts below, at and past a round of lanes.

One step's mu and forces against the oracle at the one-step bar of the parity
tests (1e-10), and the list-free sums against the walk of the stored list
bitwise: the walk subtracts every term in the list's order, whatever the
number of lanes."""
import numpy as np
import pytest

import phafd_amd as P
from helpers import make_gpu, make_oracle, rel_l2, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("style", [False, True, "linear"])
@pytest.mark.parametrize("width", [0.6, 1.0, 1.6, 1.75, 2.5])
@pytest.mark.parametrize("nchains,nbeads", [(1, 1), (1, 7), (9, 15)])
def test_force_walk_shapes(style, width, nchains, nbeads):
    w = workload(n=32, nchains=nchains, nbeads=nbeads, ljish=style, nucwidth=width, gauss_cut=3.0, zghost=1,
                 seed=31, types=2 if nbeads > 1 else 1, chain=nbeads > 1)
    g, o = make_gpu(w), make_oracle(w)
    e = make_gpu(w)
    e.set_option(P.OPT_EAGER_GRIDLIST, 1)
    e.setup(w["dt"])
    for s in (g, o, e):
        for ph in (P.PH_START, P.PH_NEIGH, P.PH_PAIR):
            s.phase(ph)
    assert rel_l2(g.get_field(P.MU), o.get_field(P.MU)) < 1e-10
    assert rel_l2(g.get_forces(), o.get_forces()) < 1e-10
    assert np.array_equal(g.get_field(P.MU), e.get_field(P.MU))
    assert np.array_equal(g.get_forces(), e.get_forces())
