"""The planes kx = 0 and kx = Nx/2 of the spectral update, updated in one kernel
with their z passes: in the bulk's launch (grids of up to 256 blocks) and in a
launch of their own, with and without thermal noise, against the FP64 run of
the separate kernels (z pass, stand-alone update, inverse z pass).

Both sides take the same modes' noise and the same update; they differ in the
rounding of a few transforms a step: 1e-11 in FP64 after four steps, and the
bar of the FP32 form (1e-6 of phi) in FP32."""
import numpy as np
import pytest

import phafd_amd as P
from helpers import rel_l2

pytestmark = pytest.mark.gpu

# (Nx, Ny, Nz): one tile of columns to many, every two-level Nz up to 256, both sides of 256 blocks
SHAPES = [(16, 16, 16), (32, 64, 16), (16, 32, 64), (32, 32, 32), (64, 64, 64), (128, 64, 64), (16, 16, 256),
          (32, 128, 128), (64, 64, 256), (128, 128, 128),
          (64, 32, 512), (32, 16, 512)]   # the planes by kernels of their own; the noise of the bulk through LDS


@pytest.mark.parametrize("noise", [P.NOISE_OFF, P.NOISE_DEVICE])
@pytest.mark.parametrize("shape", SHAPES)
def test_edge_planes(shape, noise):
    nx, ny, nz = shape
    phi = P.ic_noisy_constant((nz, ny, nx), 0.45, 0.2, 31)   # white: the edge planes carry their share of it
    out = []
    for precision, fused in ((P.FP64, 0), (P.FP64, 1), (P.FP32, 1)):
        s = P.System(nx, ny, nz, [0, 0, 0], [0.9 * nx, 1.1 * ny, 1.3 * nz], precision=precision)
        s.set_option(P.OPT_FUSE_SPECTRAL, fused)
        s.set_field(P.PHI, phi)
        s.fix_conjugate(5678, temp=1e-4, noise=noise)
        s.fix_floryhuggins(chi=2.5)
        s.setup(1e-3)
        s.run(4)
        out.append(s.get_field(P.PHI).astype(np.float64))
        s.close()
    ref, f64, f32 = out
    assert rel_l2(f64, ref) < 1e-11
    assert rel_l2(f32, ref) < 1e-6
    # the two planes by themselves: the rest of the field does not hide them
    for k in (0, nx // 2):
        a, b = (np.fft.rfft(f, axis=2)[:, :, k] for f in (f64, ref))
        if k == 0:
            a, b = a - a.mean(), b - b.mean()
        assert rel_l2(a, b) < 1e-10
