"""The mu sums of the grid-atom pass where their staging can go wrong: points
without a term, a point with more terms than one staged chunk (2048), several
chunks per block, several points per thread (grids of 2^21 points and more).
Against the walk of the stored list, bitwise: the same terms in the same order."""
import numpy as np
import pytest

import phafd_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,natoms,spread", [(32, 1, 0.0), (32, 300, 12.0), (32, 2600, 0.4), (32, 5000, 6.0),
                                             (128, 4000, 60.0), (128, 2600, 0.4)])
def test_mu_sums_bitwise(n, natoms, spread):
    rng = np.random.default_rng(natoms + n)
    xyz = n / 2 + 0.3 + spread * (rng.random((natoms, 3)) - 0.5)
    phi = P.ic_noisy_constant((n, n, n), 0.4, 0.05, 3)
    out = []
    for eager in (0, 1):
        s = P.System(n, n, n, [0, 0, 0], [float(n)] * 3, zghost=P.ZGHOST_PERIODIC)
        s.set_field(P.PHI, phi)
        s.set_atoms(xyz, np.zeros(natoms, np.int32))
        ip = s.pair_gridatom(P.PAIR_LJISH, 2.5)
        s.pair_coeff(ip, 0, 1.0, 0.1, 1.9)
        s.fix_conjugate(5678)
        s.fix_floryhuggins()
        s.neighbor(0.5)
        s.set_option(P.OPT_EAGER_GRIDLIST, eager)
        s.setup(1e-3)
        for ph in (P.PH_START, P.PH_NEIGH, P.PH_PAIR):
            s.phase(ph)
        out.append(s.get_field(P.MU))
        s.close()
    assert np.abs(out[1]).max() > 0
    assert np.array_equal(out[0], out[1])
