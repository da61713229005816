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


def _terms_in_64_bits(w, fields):
    """Forces and mu of the grid-atom styles from the FP32 fields as read back,
    and the sums of the terms' magnitudes with the kernel at its largest."""
    phi, gx, gy, gz = fields
    n, F, mu = w["n"], np.zeros((len(w["xyz"]), 3)), np.zeros_like(phi)
    Fm, mum = np.zeros(len(w["xyz"])), np.zeros_like(phi)
    grid = np.arange(n, dtype=np.float64)
    for a, (x, t) in enumerate(zip(w["xyz"], w["types"])):
        eps, phit, cs = w["eps"] * (1.0 + 0.5 * t), 0.1, w["nucwidth"] ** 2
        d = [(grid - x[c] + n / 2) % n - n / 2 for c in range(3)]
        r = (d[2][:, None, None] ** 2 + d[1][None, :, None] ** 2 + d[0][None, None, :] ** 2) / cs
        at = np.nonzero(r < 1.0)
        r = r[at]
        if w["ljish"]:
            e = np.exp(1.0 - 1.0 / (1.0 - r)) * eps
        else:
            e = (np.exp(-r / 2) - np.exp(-0.5)) * np.exp(0.5) * eps
        if w["ljish"] == "linear":
            wt, m, scale = -e, -e, np.full(r.shape, eps)
        else:
            dphi = phi[at] - phit
            wt, m, scale = 2 * dphi * e, 2 * dphi * e, 2 * np.abs(dphi) * eps
        np.add.at(mu, at, m)
        np.add.at(mum, at, scale)
        for c, g in enumerate((gx, gy, gz)):
            F[a, c] = -(g[at] * wt).sum()
        Fm[a] = (np.sqrt(gx[at] ** 2 + gy[at] ** 2 + gz[at] ** 2) * scale).sum()
    return F, mu, Fm, mum


@pytest.mark.parametrize("style", [False, True, "linear"])
@pytest.mark.parametrize("width", [0.6, 1.0, 1.6, 1.75, 2.5])
@pytest.mark.parametrize("nchains,nbeads", [(1, 1), (1, 7), (9, 15)])
def test_fp32_force_walk_shapes(style, width, nchains, nbeads):
    """The FP32 walk packs the kept terms before it adds them up.  A term's
    rounding: at most 6 units of 2^-24 of the kernel's largest value (its
    argument, exp, and the difference from its value at the cut) and 5 more of
    its factors; the Kahan sums add 2 of the terms' total."""
    w = workload(n=32, nchains=nchains, nbeads=nbeads, ljish=style, nucwidth=width, gauss_cut=3.0, zghost=1,
                 seed=31, types=2 if nbeads > 1 else 1, chain=False, lj=False)
    g = make_gpu(w, precision=P.FP32)
    for ph in (P.PH_START, P.PH_NEIGH, P.PH_PAIR):
        g.phase(ph)
    F, mu, Fm, mum = _terms_in_64_bits(w, [g.get_field(k) for k in (P.PHI, P.GRADX, P.GRADY, P.GRADZ)])
    assert width < 1 or np.abs(F).max() > 0   # a narrow kernel may hold no grid point
    assert (np.abs(g.get_forces() - F).max(1) <= 13 * 2.0 ** -24 * Fm).all()
    assert (np.abs(g.get_field(P.MU) - mu) <= 13 * 2.0 ** -24 * mum).all()
