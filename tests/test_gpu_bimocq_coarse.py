"""BIMOCQ on coarse films (needs an MI355X): the sizes on either side of the lines
between its forms (192 rows; about 50 for maps at rest), films whose flow
stretches the maps beyond the fast forms, coarse and fine films in one context, a
NaN in one of them; against the oracle."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import copy_state, load, make_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu

FIELDS = ("u_theta", "u_phi", "eta", "gamma")
# FP64: the solves' relative 1e-10 and the maps' roundings; the mixed path: FP32
# fields (6e-8 a step), u by the gradient of an FP32 Gamma. Both for six steps;
# they add up over more.
TOL = {"fp64": 1e-9, "mixed": 2e-5}


def tolerance(prec, steps):
    return TOL[prec] * max(1.0, steps / 6)


def expected(n, dt, case, steps, **kw):
    from oracle import oracle as O

    st, ua, va = case
    p = O.params(n, dt)
    ref = copy_state(st)
    O.bimocq_step(p, ref, ua, va, O.BimocqState(p, ref["eta"], ref["gamma"], blend=0.5, **kw), steps)
    return ref


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n,dt,steps", [(4, 0.05, 4), (16, 0.02, 8), (49, 0.006, 12), (64, 0.0125, 40),
                                        (101, 0.008, 25), (128, 0.006, 25), (191, 0.003, 8), (192, 0.003, 8)])
def test_either_side(prec, n, dt, steps):
    case = make_case(n, 5 + n, u_scale=1.0)
    ref = expected(n, dt, case, steps)
    with sb.SoapFilm(sb.bubble(n, dt), prec, scalar_advection="bimocq") as ctx:
        load(ctx, 0, *case)
        ctx.step(steps)
        got = ctx.state(0)
    worst = max(rel_l2(got[k], ref[k]) for k in FIELDS)
    print(f"  {prec} n={n}: {worst:.2e}", flush=True)
    assert worst <= tolerance(prec, steps), worst


@pytest.mark.parametrize("graph", [True, False])
def test_coarse_and_fine_in_one_context(graph):
    films = [(24, 0.01), (192, 0.003), (64, 0.01), (200, 0.003)]
    cases = [make_case(n, n, u_scale=1.0) for n, _ in films]
    with sb.SoapFilm([sb.bubble(n, dt) for n, dt in films], "mixed", scalar_advection="bimocq",
                     use_graph=graph) as ctx:
        for b, c in enumerate(cases):
            load(ctx, b, *c)
        ctx.step(10)
        for b, (n, dt) in enumerate(films):
            ref, got = expected(n, dt, cases[b], 10), ctx.state(b)
            worst = max(rel_l2(got[k], ref[k]) for k in FIELDS)
            assert worst <= tolerance("mixed", 10), (n, worst)


@pytest.mark.parametrize("n", [24, 64])
def test_a_nan_in_a_coarse_film(n):
    m = 2 * n
    st, ua, va = make_case(n, 3, u_scale=1.0)
    st["eta"].reshape(n, m)[n // 2, n] = np.nan
    with sb.SoapFilm(sb.bubble(n, 0.5 / n), "fp64", scalar_advection="bimocq") as ctx:
        load(ctx, 0, st, ua, va)
        ctx.advect()
        got = ctx.download(0, "eta_star").reshape(n, m)
    # the samplers skip the NaN: the advected thickness has none left
    assert np.isfinite(got).all()
