"""The sweeps of more than one species at the edges of their strips: block
heights around multiples of the 16-row strip and its four-row groups, widths
around the eight-step rounds, and species counts that leave the last compute
wave with one to four components.

Both sides evaluate the same update from the same state.  The sweeps over stored
matrices keep the order of every sum, so their result is the same; the closed
form sums in another order.  Each cell's increment is a chain of at most ni + nj
products whose factors have norm below one (diagonal dominance), so the rounding
differences add up to a small multiple of (ni + nj) eps of each component's
increments; seen, over all cases, at most 8 eps (2 x 2) to 60 eps (130 x 7), and
16 (ni + nj) eps is allowed.  An ideal gas has no DHi; a field of them of the size
of R T, which moves the species' increments by 5e-6 to 4e-3, is uploaded for the
coefficients that hold it.
"""
import numpy as np
import pytest

from shared_cfd_amd import cases as C
from shared_cfd_amd import chem
from shared_cfd_amd.native import OPT_JVP_SWEEP, OPT_SKEW_SWEEP, Solver

from chem_cases import NO27, no27_plus_inert

pytestmark = pytest.mark.gpu


SIZES = [(2, 2, 2), (2, 14, 17), (3, 13, 4), (4, 15, 15), (5, 14, 5), (8, 30, 16), (9, 31, 17), (9, 6, 48),
         (9, 22, 49), (10, 3, 65), (11, 130, 7), (12, 9, 34), (13, 62, 33), (14, 33, 20), (16, 21, 33)]


def _increments(case, skew, reps, jvp=1, dhi=0.0):
    s = Solver(case)
    s.set_option(OPT_SKEW_SWEEP, skew)
    s.set_option(OPT_JVP_SWEEP, jvp)
    s.prepare()
    rng = np.random.default_rng(9)
    for b in range(case.nblocks if dhi else 0):  # a step keeps all but the first species' DHi
        s.upload("DHI", b, rng.uniform(-dhi, dhi, (case.nj[b] + 4, case.ni[b] + 4, case.ny)))
    for k in range(reps):
        s.step(k + 1, 0)
    out = [s.download("Q", b)[2:-2, 2:-2] - case.q0[b][2:-2, 2:-2] for b in range(case.nblocks)]
    s.close()
    return out


@pytest.mark.parametrize("dhi", [0.0, 3e4])
@pytest.mark.parametrize("scheme", [C.SCHEME_LUSGS, C.SCHEME_NR])
@pytest.mark.parametrize("ny,ni,nj", SIZES)
def test_strip_edges(scheme, ny, ni, nj, dhi):
    case = C.random_case(seed=ni + nj, ni=(ni, 9), nj=(nj, 20), ny=ny, scheme=scheme)
    case.params.res_rate_warning = case.params.res_rate_error = 1e300
    eps = np.finfo(float).eps
    for k, (a, b) in enumerate(zip(_increments(case, 1, 2, dhi=dhi), _increments(case, 0, 2, dhi=dhi))):
        scale = np.max(np.abs(b), axis=(0, 1))
        assert np.all(scale > 0.0)
        assert np.all(np.max(np.abs(a - b), axis=(0, 1)) <= 16 * (case.ni[k] + case.nj[k]) * eps * scale)


@pytest.mark.parametrize("scheme", [C.SCHEME_LUSGS, C.SCHEME_PRECON_LUSGS, C.SCHEME_PRECON])
@pytest.mark.parametrize("ny,ni,nj", SIZES)
def test_strip_edges_stored_matrices(scheme, ny, ni, nj):
    local = scheme != C.SCHEME_LUSGS
    case = C.random_case(seed=ni + nj, ni=(ni, 9), nj=(nj, 20), ny=ny, scheme=scheme, time_step=1 if local else 0,
                         mach=0.3)
    case.params.res_rate_warning = case.params.res_rate_error = 1e300
    for a, b in zip(_increments(case, 1, 2, jvp=0), _increments(case, 0, 2)):
        assert np.max(np.abs(b)) > 0.0
        assert np.array_equal(a, b)


@pytest.mark.parametrize("inert", [0, 1, 4, 8])
def test_closed_form_with_a_mechanism(tmp_path, inert):
    """One step of a disturbed mixing layer: every species' DHi, the first's too,
    from the thermodynamics, which both sides evaluate on the same state."""
    ns = 8 + inert
    lm = chem.parse(no27_plus_inert(str(tmp_path), inert)[0] if inert else NO27)
    rng = np.random.default_rng(ns)
    fuel, ox = rng.uniform(0.01, 0.1, ns), rng.uniform(0.01, 0.1, ns)
    case = C.mixing_layer(lm, ni=31, nj=33, reaction=0, fuel=fuel / fuel.sum(), ox=ox / ox.sum())
    case.q0[0] = case.q0[0] * (1.0 + 0.1 * rng.random(case.q0[0].shape[:2]))[..., None]
    a, b = _increments(case, 1, 1)[0], _increments(case, 0, 1)[0]
    scale = np.max(np.abs(b), axis=(0, 1))
    assert np.all(scale > 0.0)
    assert np.all(np.max(np.abs(a - b), axis=(0, 1)) <= 16 * (31 + 33) * np.finfo(float).eps * scale)
