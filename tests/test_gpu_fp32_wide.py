"""The FP32 passes of 512 lines.  The z update of a followed step takes 16 lines
per block, the x c2r 32 where Ny holds them and 16 otherwise: the step against
FP64 at the bar of the FP32 form (phi 1e-6 of the FP64 run)."""
import numpy as np
import pytest

import phafd_amd as P
from helpers import rel_l2

pytestmark = pytest.mark.gpu


# Ny = 16: one z block per plane; Nx = 512: 16 rows per x block, 32 need Ny >= 32
@pytest.mark.parametrize("shape", [(64, 16, 512), (64, 32, 512), (32, 64, 512), (512, 16, 32), (512, 32, 64),
                                   (512, 32, 512)])
def test_fp32_steps(shape):
    nx, ny, nz = shape
    phi = P.ic_noisy_constant((nz, ny, nx), 0.45, 0.1, 7)
    out = []
    for prec in (P.FP64, P.FP32):
        s = P.System(nx, ny, nz, [0, 0, 0], [float(v) for v in shape], precision=prec)
        s.set_field(P.PHI, phi)
        s.fix_conjugate(5678)
        s.fix_floryhuggins(chi=2.5)
        s.setup(1e-3)
        s.run(4)
        out.append([s.get_field(w) for w in (P.PHI, P.GRADX, P.GRADY, P.GRADZ)])
        s.close()
    assert rel_l2(out[1][0], out[0][0]) < 1e-6
    for a, b in zip(out[1][1:], out[0][1:]):
        assert rel_l2(a, b) < 1e-4
