"""The one-launch fold of ghost forces where an atom's image lists can go
wrong: beads in the corners of the box (seven images), on its edges and faces,
none near a face, one bead, no z images, and a box too small for disjoint swaps
(the swap-by-swap folds).  Forces against the oracle at the one-step bar."""
import numpy as np
import pytest

import phafd_amd as P
from helpers import apply, rel_l2
from oracle import oracle_ctypes as O

pytestmark = pytest.mark.gpu


def _beads(kind, box, rng):
    if kind == "one":
        return np.full((1, 3), 0.3 * box)
    if kind == "corner":   # close pairs across all three faces
        return (rng.random((40, 3)) - 0.5) * 1.6 % box
    if kind == "edges":    # two coordinates at a face, the third anywhere
        x = rng.random((60, 3)) * box
        x[:, :2] = (rng.random((60, 2)) - 0.5) * 2.0 % box
        return np.concatenate([x, x[:, [1, 2, 0]]])
    if kind == "inside":
        return box / 2 + (rng.random((50, 3)) - 0.5) * 4.0
    return rng.random((400, 3)) * box


@pytest.mark.parametrize("zghost", [0, 1])
@pytest.mark.parametrize("kind,n,box", [("one", 16, 16.0), ("corner", 16, 16.0), ("edges", 32, 32.0),
                                        ("inside", 16, 16.0), ("all", 32, 32.0), ("all", 16, 8.0), ("corner", 8, 6.0),
                                        ("corner", 8, 4.0), ("all", 16, 4.0)])   # the last two: swaps that share atoms
def test_forces_of_folded_images(kind, n, box, zghost):
    rng = np.random.default_rng(n)
    xyz = _beads(kind, box, rng)
    w = dict(n=n, box=box, origin=0.0, phi=P.ic_noisy_constant((n, n, n), 0.4, 0.1, 5), xyz=xyz,
             mol=np.zeros(len(xyz), np.int32), types=np.zeros(len(xyz), np.int32), ntypes=1, chi=2.5, gauss_cut=2.0,
             nucwidth=1.6, ljish=True, lj=False, chain=False, drag=False, skin=0.4, dt=1e-3, zghost=zghost, noise=0,
             eps=1.0, harmonic=(1.2, 5.0), starts=np.zeros(0, np.int32), ends=np.zeros(0, np.int32))
    g = apply(P.System(n, n, n, [0, 0, 0], [box] * 3, zghost=zghost), w, False)
    o = apply(O.System(n, n, n, [0, 0, 0], [box] * 3, zghost=zghost), w, True)
    for s in (g, o):
        for ph in (P.PH_START, P.PH_NEIGH, P.PH_PAIR):
            s.phase(ph)
    assert rel_l2(g.get_forces(), o.get_forces()) < 1e-10


@pytest.mark.parametrize("zghost", [0, 1])
@pytest.mark.parametrize("kind,n,box", [("corner", 16, 16.0), ("edges", 32, 32.0), ("all", 32, 32.0), ("all", 16, 8.0),
                                        ("corner", 16, 4.0)])   # the last: images along both ways, no one-launch fold
def test_folded_sums_are_the_swaps_bitwise(kind, n, box, zghost):
    """lj/cut forces (products and quotients only, no function whose rounding
    is the library's own) folded image by image in the oracle, swap after swap:
    the same sums in the same order give the same bits."""
    rng = np.random.default_rng(n + 1)
    xyz = _beads(kind, box, rng)
    out = []
    for M, gpu in ((P, True), (O, False)):
        s = M.System(n, n, n, [0, 0, 0], [box] * 3, zghost=zghost)
        s.set_field(P.PHI, P.ic_noisy_constant((n, n, n), 0.4, 0.1, 5))
        s.set_atoms(xyz, np.zeros(len(xyz), np.int32), tags=np.arange(len(xyz), dtype=np.int32),
                    mols=np.zeros(len(xyz), np.int32))
        if gpu:
            s.pair_ljcut(2.0, 1.0, 1.0)
        else:
            s.add_pair(O.PAIR_LJCUT, 2.0, 1.0, 1.0)
        s.fix_conjugate(5678, 1.0, 1.0, 1.0, 1.0, 0)
        s.neighbor(0.4)
        s.setup(1e-3)
        for ph in (P.PH_START, P.PH_NEIGH, P.PH_PAIR):
            s.phase(ph)
        out.append(s.get_forces())
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(*out)
