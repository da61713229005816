"""The y and z derivatives taken of phi's own lines, and their Nyquist terms,
where their tiles can go wrong: axis lengths of every two-level split, planes
with fewer rows than a tile, columns of several planes in one tile.

The fields are white noise, so the Nyquist modes carry as much as any other.
Gradient of the first step (from phi) and of a later one (from the updated
spectrum) against the oracle at the bar of the spectral tests (1e-12)."""
import numpy as np
import pytest

import phafd_amd as P
from helpers import rel_l2
from oracle import oracle_ctypes as O

pytestmark = pytest.mark.gpu

SHAPES = [(64, 256, 32), (32, 64, 256), (64, 512, 16), (1024, 32, 16), (128, 64, 64), (256, 16, 128), (512, 32, 32),
          (32, 512, 32), (64, 64, 128), (32, 32, 512)]   # (Nx, Ny, Nz), all above 2^18 points


@pytest.mark.parametrize("shape", SHAPES)
def test_line_gradient(shape):
    nx, ny, nz = shape
    assert nx * ny * nz > 1 << 18
    period = [0.9 * nx, 1.1 * ny, 1.3 * nz]
    phi = P.ic_noisy_constant((nz, ny, nx), 0.45, 0.2, 77)
    out = []
    for M in (P, O):
        s = M.System(nx, ny, nz, [0, 0, 0], period)
        s.set_field(P.PHI, phi)
        s.fix_conjugate(5678, 1.0, 1.0, 1.0, 1.0, 0)
        s.fix_floryhuggins(1.0, 1.0, 2.5)
        s.setup(1e-3)
        out.append(s)
    g, o = out
    for s in (g, o):
        s.phase(P.PH_START)
    for w in (P.GRADX, P.GRADY, P.GRADZ):
        assert rel_l2(g.get_field(w), o.get_field(w)) < 1e-12
    for s in (g, o):
        s.run(3)   # the last step's gradient comes from the step before it
    for w in (P.GRADX, P.GRADY, P.GRADZ, P.PHI):
        assert rel_l2(g.get_field(w), o.get_field(w)) < 1e-12


@pytest.mark.parametrize("shape", SHAPES + [(32, 64, 16), (64, 32, 16), (32, 64, 64), (128, 128, 128), (16, 8, 32)])
def test_stateless_gradient(shape):
    """phafd_hip_gradphi: the line kernels with the Nyquist terms from the
    alternating sums (16 x 8 x 32: the transforms)."""
    nx, ny, nz = shape
    period = [0.9 * nx, 1.1 * ny, 1.3 * nz]
    phi = P.ic_noisy_constant((nz, ny, nx), 0.45, 0.2, 78)
    for a, b in zip(P.gradphi(phi, period), O.gradphi(phi, period)):
        assert rel_l2(a, b) < 1e-12


@pytest.mark.parametrize("shape", [(32, 16, 16), (64, 32, 64), (128, 128, 128), (16, 8, 32)])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_stateless_gradient_of_a_field_with_a_hole(shape, value):
    """One NaN or infinity in phi, at the first, the last and an inner point:
    nothing of the gradient is finite, as after a transform in three dimensions
    (16 x 8 x 32)."""
    nx, ny, nz = shape
    phi = P.ic_noisy_constant((nz, ny, nx), 0.45, 0.2, 79)
    for at in ((0, 0, 0), (nz - 1, ny - 1, nx - 1), (nz // 2 + 1, 5, 3)):
        bad = phi.copy()
        bad[at] = value
        for g in P.gradphi(bad, [1.0 * nx, 1.0 * ny, 1.0 * nz]):
            assert not np.isfinite(g).any()
