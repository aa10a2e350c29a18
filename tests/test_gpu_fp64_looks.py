"""The host-driven PCG's looks at its flags (needs an MI355X): a step that needs far
fewer iterations than the one before, after a change of the step size or a new
film, does not run the old count's launches; results against the oracle."""
import time

import numpy as np
import pytest

import soapbubble_amd as sb
from cases import copy_state, load, make_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("by", ["set_dt", "upload"])
def test_no_launches_of_an_older_solve(by):
    """218 iterations, then 2: with the old count's launches the first step takes
    six times as long as the next ones."""
    n = 256
    hard, easy = 0.2, 0.0005
    st, ua, va = make_case(n, 3)
    still = {"u_theta": 0 * st["u_theta"], "u_phi": 0 * st["u_phi"], "eta": np.ones_like(st["eta"]),
             "gamma": np.ones_like(st["gamma"])}
    first, later = [], []
    with sb.SoapFilm(sb.bubble(n, hard, airflow=by == "set_dt"), "fp64") as ctx:
        for _ in range(5):
            if by == "set_dt":
                ctx.set_dt(hard)
            load(ctx, 0, st, ua, va)
            ctx.step(2)
            assert ctx.stats(0)["iterations"] > 100
            if by == "set_dt":
                ctx.set_dt(easy)
            else:
                # an even film at rest without air: nothing to solve
                load(ctx, 0, still, ua, va)
            times = []
            for _ in range(4):
                t0 = time.perf_counter()
                ctx.step(1)
                times.append(time.perf_counter() - t0)
            assert ctx.stats(0)["iterations"] < 10
            first.append(times[0])
            later.append(np.median(times[1:]))
    f, g = np.median(first), np.median(later)
    print(f"  after {by}: first step {1e6 * f:.0f} us, later ones {1e6 * g:.0f}", flush=True)
    assert f < 3 * g, (f, g)


def test_results():
    """Solves of many and of few iterations in turn (each leaves 1e-10 of |b|)."""
    from oracle import oracle as O

    n, dts = 48, (0.1, 0.001, 0.1)
    st, ua, va = make_case(n, 9, u_scale=0.3)
    ref = copy_state(st)
    with sb.SoapFilm(sb.bubble(n, dts[0]), "fp64", advance_time=False) as ctx:
        load(ctx, 0, st, ua, va)
        for dt in dts:
            ctx.set_dt(dt)
            ctx.step(2)
            p = O.params(n, dt)
            O.step(p, ref, ua, va, 2, advance_time=False)
        got, s = ctx.state(0), ctx.stats(0)
    assert s["failed_solves"] == 0, s
    for k in ref:
        assert rel_l2(got[k], ref[k]) < 1e-8, (k, rel_l2(got[k], ref[k]))
