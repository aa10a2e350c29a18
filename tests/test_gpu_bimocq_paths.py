"""The BIMOCQ kernels' two forms (needs an MI355X): smooth maps and coarse ones
whose neighbours are too far apart for the series, rows of any length, the
polar rows, one and five samples, maps carried a large angle, and a film with
a NaN, against the oracle."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import copy_state, load, make_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu

FIELDS = ("u_theta", "u_phi", "eta", "gamma")


# FP64: the solves' relative 1e-10 and the maps' roundings over a few steps; the
# mixed path: FP32 fields (6e-8 a step), u by the gradient of an FP32 Gamma.
TOL = {"fp64": 1e-9, "mixed": 2e-5}


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("multisample", [True, False])
@pytest.mark.parametrize("n,dt,steps", [(12, 0.02, 5), (49, 0.01, 6), (64, 0.01, 6), (101, 0.005, 6),
                                        (128, 0.12, 3)])
def test_bimocq_steps(prec, multisample, n, dt, steps):
    from oracle import oracle as O

    st, ua, va = make_case(n, 17 + n, u_scale=1.0)
    p = O.params(n, dt)
    ref = copy_state(st)
    b = O.BimocqState(p, ref["eta"], ref["gamma"], blend=0.4, multisample=multisample)
    O.bimocq_step(p, ref, ua, va, b, steps)
    with sb.SoapFilm(sb.bubble(n, dt), prec, scalar_advection="bimocq", blend=0.4,
                     multisample=multisample) as ctx:
        load(ctx, 0, st, ua, va)
        ctx.step(steps)
        got, s = ctx.state(0), ctx.stats(0)
    worst = max(rel_l2(got[k], ref[k]) for k in FIELDS)
    print(f"  {prec} n={n} dt={dt} samples={5 if multisample else 1}: {worst:.2e} distortion "
          f"{s['distortion']:.3f}", flush=True)
    assert worst <= TOL[prec], worst


def test_a_nan_takes_the_skipping_samplers():
    n, m, dt = 64, 128, 0.01
    st, ua, va = make_case(n, 3, u_scale=1.0)
    st["eta"].reshape(n, m)[40, 100] = np.nan
    with sb.SoapFilm(sb.bubble(n, dt), "fp64", scalar_advection="bimocq") as ctx:
        load(ctx, 0, st, ua, va)
        ctx.advect()
        got = ctx.download(0, "eta_star").reshape(n, m)
    # the samplers skip the NaN: the advected thickness has none left
    assert np.isfinite(got).all()
    assert abs(got[40, 100] - 1.0) < 0.3
