"""The spectral preconditioner of the automatic inner method in the stiff regime
(needs an MI355X): rows of any length and ensembles against the oracle, the
exact case of an even film, and the hand-over to multigrid for a film too
uneven for it."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import copy_state, load, make_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu

FIELDS = ("u_theta", "u_phi", "eta", "gamma")
RADIUS = 0.05

# The mixed path's distance from the oracle after a few steps in this regime:
# the FP32 fields' rounding (6e-8) grown by the steps and, in u, by the
# gradient of an FP32 Gamma over a cell (n / pi <= 100 of them, times dt M of
# about 0.1): 1e-6 at most; a solve that met its tolerance adds 1e-10 of that.
TOL = 5e-6


def stiff_dt(n):
    """A step that is stiff on n rows: mu grows with (n dt)^2."""
    return 0.005 * 256 / n


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("n", [16, 33, 64, 100, 250, 272])
def test_stiff_films(n, graph):
    from oracle import oracle as O

    st, ua, va = make_case(n, 31 + n, u_scale=0.1)
    dt = stiff_dt(n)
    with sb.SoapFilm(sb.bubble(n, dt, radius=RADIUS), "mixed", use_graph=graph) as ctx:
        load(ctx, 0, st, ua, va)
        ctx.step(9)
        got, s = ctx.state(0), ctx.stats(0)
    print(f"  n={n} iterations {s['iterations']} refinements {s['outer']}", flush=True)
    assert s["failed_solves"] == 0 and s["max_residual"] <= 1e-10, s
    ref = copy_state(st)
    O.step(O.params(n, dt, radius=RADIUS), ref, ua, va, 9)
    for k in FIELDS:
        assert rel_l2(got[k], ref[k]) < TOL, (k, rel_l2(got[k], ref[k]))


def test_stiff_ensemble():
    from oracle import oracle as O

    sizes = [48, 100, 128]
    cases = [make_case(n, 60 + n, u_scale=0.1) for n in sizes]
    with sb.SoapFilm([sb.bubble(n, stiff_dt(n), radius=RADIUS) for n in sizes], "mixed",
                     use_graph=True) as ctx:
        for b, (st, ua, va) in enumerate(cases):
            load(ctx, b, st, ua, va)
        ctx.step(11)
        for b, (n, (st, ua, va)) in enumerate(zip(sizes, cases)):
            assert ctx.stats(b)["failed_solves"] == 0
            ref = copy_state(st)
            O.step(O.params(n, stiff_dt(n), radius=RADIUS), ref, ua, va, 11)
            got = ctx.state(b)
            for k in FIELDS:
                assert rel_l2(got[k], ref[k]) < TOL, (n, k)


def test_even_film_is_solved_at_once():
    """With constant thickness and concentration the row-mean operator is the
    operator itself: an FP32 application solves to its rounding, so each
    refinement needs an iteration or two."""
    n = 128
    N = n * 2 * n
    st = {"u_theta": np.zeros(N - 2 * n), "u_phi": np.zeros(N), "eta": np.full(N, 0.5),
          "gamma": np.ones(N)}
    _, ua, va = make_case(n, 4)
    with sb.SoapFilm(sb.bubble(n, stiff_dt(n), radius=RADIUS), "mixed") as ctx:
        load(ctx, 0, st, ua, va)
        ctx.step(1)
        s = ctx.stats(0)
    print("  iterations", s["iterations"], "refinements", s["outer"], flush=True)
    assert s["failed_solves"] == 0
    assert s["iterations"] <= 2 * (s["outer"] - 1), s


@pytest.mark.parametrize("thick", [4.0, 30.0])
@pytest.mark.parametrize("graph", [True, False])
def test_uneven_films(graph, thick):
    """A film hundreds of times thinner in places, with face weights (1 / (eta +
    Cr dt)) ten and seventy times apart, on either side of the line to
    multigrid: from the start, and uploaded into a running context that had
    the spectral preconditioner's schedule for an even film."""
    from oracle import oracle as O

    n, dt = 64, stiff_dt(64)
    st, ua, va = make_case(n, 8, u_scale=0.1)
    thin = copy_state(st)
    th = (np.arange(n) + 0.5) * np.pi / n
    ph = np.arange(2 * n) * np.pi / n
    w = 0.5 + 0.5 * np.sin(th)[:, None] * np.cos(ph)[None]
    thin["eta"] = (0.01 + thick * w ** 4).ravel()
    for first in (None, st):
        with sb.SoapFilm(sb.bubble(n, dt, radius=RADIUS), "mixed", use_graph=graph) as ctx:
            if first is not None:
                load(ctx, 0, first, ua, va)
                ctx.step(12)
            load(ctx, 0, thin, ua, va)
            ctx.set_time(0.0)
            ctx.step(9)
            got, s = ctx.state(0), ctx.stats(0)
        assert s["failed_solves"] == 0, s
        ref = copy_state(thin)
        O.step(O.params(n, dt, radius=RADIUS), ref, ua, va, 9)
        for k in FIELDS:
            assert rel_l2(got[k], ref[k]) < 5e-5, (k, rel_l2(got[k], ref[k]))
