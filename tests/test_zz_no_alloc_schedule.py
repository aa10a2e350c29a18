"""The solve schedule of sf_step_noalloc (needs an MI355X): weakly to strongly
coupled systems, whose first refinement meets the tolerance or is followed by
the full schedule, against sf_step; and the schedule a caller fixes."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import make_case
from conftest import rel_l2
from test_zz_no_alloc import FIELDS, _Hip, _noalloc, _reference

pytestmark = pytest.mark.gpu

# Both runs' solves leave 1e-10 of |b|; beyond that their FP32 fields differ by
# roundings (6e-8) carried through a few steps: well below 2e-6.
TOL = 2e-6


@pytest.mark.parametrize("n", [20, 64, 101])
@pytest.mark.parametrize("dt", [0.0005, 0.01, 0.04])
def test_schedules_match_sf_step(n, dt):
    hip = _Hip()
    st, ua, va = make_case(n, 3 * n, u_scale=0.5)
    want, _ = _reference(n, dt, st, ua, va, 5)
    got, gs = _noalloc(hip, n, dt, st, ua, va, 5, False)
    print(f"  n={n} dt={dt}: {gs['iterations']} iterations, {gs['outer']} refinements", flush=True)
    assert gs["failed_solves"] == 0 and gs["max_residual"] <= 1e-10, gs
    for k in FIELDS:
        assert rel_l2(got[k], want[k]) < TOL, (k, rel_l2(got[k], want[k]))
    hip.free()


def test_a_fixed_schedule_stays_fixed():
    hip = _Hip()
    n, dt = 64, 0.005
    st, ua, va = make_case(n, 9, u_scale=0.5)
    ins = [hip.put(st[k]) for k in FIELDS]
    air = [hip.put(ua), hip.put(va)]
    outs = [hip.put(np.full(sz, np.nan)) for _, sz in ins]
    s = sb.step_noalloc(sb.bubble(n, dt), sb.options("mixed", max_outer=1, max_inner=7), 0.0, 1,
                        [p for p, _ in ins], [p for p, _ in air], [p for p, _ in outs])
    assert s["iterations"] == 7, s
    hip.free()
