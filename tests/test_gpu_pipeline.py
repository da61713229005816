"""Runs whose next step is enqueued before the step ahead of it is checked."""
import numpy as np
import pytest

import phafd_amd as P
from helpers import apply, workload

pytestmark = pytest.mark.gpu


def _system(integrator, precision=P.FP64, n=16, box=None, dt=1e-3, **kw):
    w = workload(n=n, box=box, nchains=3, nbeads=7, seed=8, var=0.05, zghost=1, dt=dt, chain=False, **kw)
    s = apply(P.System(n, n, n, [0] * 3, [w["box"]] * 3, zghost=1, precision=precision), w, False, setup=False)
    # "both": one fix moves the first chain, the other the rest
    a, b = (1, 1) if integrator == "both" else (3, 0)
    if integrator in ("chain", "both"):   # soft enough for the time step of the unstable runs
        s.fix_chain(w["starts"][:a], w["ends"][:a], 1.0, 20.0, 1.0, 1.0)
    if integrator in ("drag", "both"):
        s.fix_drag(w["starts"][b:], w["ends"][b:], 1.0)
    if integrator == "rods":
        s.fix_semiflexible(1, w["starts"], w["ends"], 99, 1.0, 0.5, 1.0, 2.0, 1.0)
    s.set_option(P.OPT_NEXT_GRADIENT, 0)   # the same arithmetic in the last step of a run as in the others
    s.setup(dt)
    return s, w


def _until_nan(s, step, most=100):
    """Runs of `step` steps until one reports NaN; the steps done before that run."""
    for k in range(0, most, step):
        try:
            s.run(step)
        except P.PhafdError as e:
            assert e.code == -3
            return k
    raise AssertionError("no NaN")


@pytest.mark.parametrize("integrator", ["drag", "rods", "chain", "both"])
@pytest.mark.parametrize("precision,n,box", [(P.FP64, 16, None), (P.FP32, 16, None), (P.FP64, 16, 8.0), (P.FP64, 8, None)])
def test_atoms_after_a_nan_are_those_of_its_step(integrator, precision, n, box):
    """A run that ends in NaN leaves the positions, the forces and the bead-rod
    noise of the step reported, whether or not a step was enqueued behind it
    (box 8: too small for the one-launch fold; n = 8: no fused passes).  The
    time step makes the explicit update unstable."""
    dt = 4e-3 * ((n if box is None else box) / n) ** 4
    a, w = _system(integrator, precision, n, box, dt)
    b, _ = _system(integrator, precision, n, box, dt)
    assert _until_nan(a, 100) == 0
    assert _until_nan(b, 1) >= 2
    for x, y in zip(a.get_atoms() + (a.get_forces(),), b.get_atoms() + (b.get_forces(),)):
        assert np.isfinite(x).all()
        assert np.array_equal(x, y)
    for s in (a, b):   # and the runs go on alike with a field that is whole
        s.set_field(P.PHI, w["phi"])
        s.setup(dt)
        s.run(4)
    for x, y in zip(a.get_atoms() + (a.get_forces(),), b.get_atoms() + (b.get_forces(),)):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("n,precision", [(16, P.FP64), (16, P.FP32), (64, P.FP64), (128, P.FP64)])
def test_nan_of_a_followed_step_is_reported(n, precision):
    """phi(0,0,0) as the kernels publish it where the next step's gradient is
    made with the update: through spectra, and (128) from phi's lines."""
    s, _ = _system("chain", precision, n, dt=4e-3)
    s.set_option(P.OPT_NEXT_GRADIENT, 1)
    assert _until_nan(s, 100) == 0
    for x in s.get_atoms() + (s.get_forces(),):
        assert np.isfinite(x).all()


@pytest.mark.parametrize("integrator", ["drag", "rods", "chain", "both"])
@pytest.mark.parametrize("precision", [P.FP64, P.FP32])
@pytest.mark.parametrize("fuse_fh", [0, 1])
def test_a_run_is_its_steps_one_by_one(integrator, precision, fuse_fh):
    """Steps enqueued ahead, decisions and flags read mid-step (published by
    the r2c of mu, or copied), both halves of the integrators together:
    bitwise the same as runs of one step, through list rebuilds."""
    a, _ = _system(integrator, precision, 32, skin=0.05)
    b, _ = _system(integrator, precision, 32, skin=0.05)
    for s in (a, b):
        s.set_option(P.OPT_FUSE_FH, fuse_fh)
    for _ in range(3):
        a.run(20)
        for _ in range(20):
            b.run(1)
        for x, y in zip(a.get_atoms() + (a.get_forces(), a.get_field(P.PHI)),
                        b.get_atoms() + (b.get_forces(), b.get_field(P.PHI))):
            assert np.array_equal(x, y)
        assert a.counts() == b.counts()
    assert a.counts()["ncalls"] > 2


@pytest.mark.parametrize("integrator", ["drag", "both"])
def test_halves_together_are_the_halves_in_their_places(integrator):
    """run() takes both halves of an atom integrator at initial_integrate; the
    hooks one by one take the second at final_integrate.  Without Flory-Huggins
    and transforms fused the fields' arithmetic is the hooks' own."""
    a, _ = _system(integrator, skin=0.05)
    b, _ = _system(integrator, skin=0.05)
    for s in (a, b):
        s.set_option(P.OPT_FUSE_FH, 0)
        s.set_option(P.OPT_FUSE_SPECTRAL, 0)
    a.run(12)
    for _ in range(12):
        for ph in (P.PH_START, P.PH_NEIGH, P.PH_PAIR, P.PH_INITIAL, P.PH_POSTFORCE, P.PH_PREFINAL, P.PH_FINAL,
                   P.PH_POSTFINAL):
            b.phase(ph)
    for x, y in zip(a.get_atoms() + (a.get_forces(), a.get_field(P.PHI)),
                    b.get_atoms() + (b.get_forces(), b.get_field(P.PHI))):
        assert np.array_equal(x, y)
