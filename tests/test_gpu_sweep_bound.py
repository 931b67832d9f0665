"""The bounded wait of the sweeps' hand-off: with the smallest bound every strip
but the first gives up after three looks (about 2 us), before its neighbour's
columns arrive (a strip's edge row runs 18 steps behind its first row, and the
sweep's first loads come before that), feeds zeros to its own sweep and runs to
its end, so each kernel of the step exits and the step returns SHCFD_E_SPIN.
With the default bound the same context then gives the result of a fresh one,
bit for bit.
"""
import numpy as np
import pytest

from shared_cfd_amd import cases as C
from shared_cfd_amd.native import OPT_JVP_SWEEP, OPT_SPIN_LIMIT, ShcfdError, Solver

pytestmark = pytest.mark.gpu

E_SPIN = 9
TALL = ((40, 9), (190, 33))          # 12 and 3 strips
MANY = ((20,) * 100, (60,) * 100)    # 4 strips each: more strips than CUs


def _solver(case, jvp):
    s = Solver(case)
    s.set_option(OPT_JVP_SWEEP, jvp)
    s.snapshot_save(0, "Q")
    return s


def _step(s):
    s.snapshot_load(0, "Q")
    s.set_time(0.0, True)
    s.prepare()
    s.step(1, 0)
    return [s.download("Q", b)[2:-2, 2:-2] for b in range(s.case.nblocks)]


@pytest.mark.parametrize("ny,scheme,jvp,blocks", [
    (1, C.SCHEME_LUSGS, 1, TALL), (1, C.SCHEME_PRECON_LUSGS, 1, TALL), (1, C.SCHEME_DUAL, 1, TALL),
    (1, C.SCHEME_LUSGS, 1, MANY), (1, C.SCHEME_DUAL, 1, MANY),
    (2, C.SCHEME_LUSGS, 1, TALL), (9, C.SCHEME_LUSGS, 1, TALL), (9, C.SCHEME_NR, 1, TALL), (16, C.SCHEME_LUSGS, 1, TALL),
    (9, C.SCHEME_LUSGS, 0, TALL), (9, C.SCHEME_PRECON_LUSGS, 1, TALL), (16, C.SCHEME_PRECON, 1, TALL)])
def test_expired_wait_is_an_error_and_leaves_the_context_usable(ny, scheme, jvp, blocks):
    local = scheme in (C.SCHEME_PRECON_LUSGS, C.SCHEME_PRECON)
    case = C.random_case(seed=5, ni=blocks[0], nj=blocks[1], ny=ny, scheme=scheme, time_step=1 if local else 0, mach=0.3)
    case.params.res_rate_warning = case.params.res_rate_error = 1e300
    fresh, s = _solver(case, jvp), _solver(case, jvp)
    want = _step(fresh)
    fresh.close()
    s.set_option(OPT_SPIN_LIMIT, 1)
    with pytest.raises(ShcfdError) as e:
        _step(s)
    assert e.value.code == E_SPIN
    s.set_option(OPT_SPIN_LIMIT, 1 << 23)
    for a, b in zip(_step(s), want):
        assert np.all(np.isfinite(b)) and np.array_equal(a, b)
    s.close()
