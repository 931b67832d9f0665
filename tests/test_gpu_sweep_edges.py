"""The optimised LU-SGS sweeps at the edges of their strips: block heights
around multiples of the 16-row strip and its four-row groups, widths around
the padding of the step count, and more strips than a CU each.

Both sides evaluate the same update from the same state; the optimised one
folds the operators and orders its sums differently.  Each cell's increment
is a chain of at most ni + nj products whose factors have norm below one
(diagonal dominance), so the rounding differences add up to a small multiple
of (ni + nj) eps of the increments: below 1e-12 here.
"""
import numpy as np
import pytest

from shared_cfd_amd import cases as C
from shared_cfd_amd.native import Solver

pytestmark = pytest.mark.gpu


def _increments(case, fast):
    s = Solver(case, fast=fast)
    s.prepare()
    s.iterate(1, 2, 0)
    out = [s.download("Q", b)[2:-2, 2:-2] - case.q0[b][2:-2, 2:-2] for b in range(case.nblocks)]
    s.close()
    return out


@pytest.mark.parametrize("scheme", [C.SCHEME_LUSGS, C.SCHEME_DUAL, C.SCHEME_PRECON_LUSGS])
@pytest.mark.parametrize("ni,nj", [(2, 2), (13, 4), (14, 5), (15, 15), (30, 16), (31, 17), (46, 33), (62, 48), (3, 65),
                                   (130, 7)])
def test_strip_edges(scheme, ni, nj):
    case = C.random_case(seed=ni + nj, ni=(ni, 9), nj=(nj, 20), scheme=scheme,
                         time_step=1 if scheme == C.SCHEME_PRECON_LUSGS else 0)
    for a, b in zip(_increments(case, True), _increments(case, False)):
        assert np.max(np.abs(b)) > 0.0
        for k in range(4):
            assert np.max(np.abs(a[..., k] - b[..., k])) <= 1e-12 * max(np.max(np.abs(b[..., k])), 1e-300), k


@pytest.mark.parametrize("scheme", [C.SCHEME_LUSGS, C.SCHEME_DUAL])
def test_two_strips_per_cu(scheme):
    """More strips than CUs: the schedule that shares a CU between strips."""
    n = 300
    case = C.random_case(seed=3, ni=(5,) * n, nj=(18,) * n, scheme=scheme)
    for a, b in zip(_increments(case, True), _increments(case, False)):
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))
