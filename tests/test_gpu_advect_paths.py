"""The advection kernel's variants against the oracle (needs an MI355X): one
trace a block and all three, rows of any length, tiles narrower than a wave,
the two polar rows, traces across a pole, and steps from a fraction of a cell
to a large part of the sphere (the series and the general form of a trace's
legs)."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import make_case, load

pytestmark = pytest.mark.gpu

FIELDS = ("u_theta", "u_phi", "eta", "gamma")


# Tolerance, largest difference over the field's largest value. A field of
# degree <= 6 changes by at most about 12 times its largest value a radian, and
# a traced angle is a few roundings of the precision off the exact one: eight
# of them are 8 * 2^-24 * 12 = 6e-6 in FP32 (whose polynomial atan2 adds 1.2e-7
# rad: 1.5e-6), plus the rounding of the field itself. The FP64 paths' angles
# come from acos near the poles in the oracle, whose error is a rounding over
# sin(theta) >= pi / (2 n): 2^-53 * 1024 * 12 = 1e-12, times eight.
TOL = {"fp64": 1e-11, "mixed": 1e-5}


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [4, 6, 16, 33, 64, 101, 128, 250, 512, 544])
@pytest.mark.parametrize("move", [0.002, 0.05, 0.4])
def test_advection(prec, n, move):
    from oracle import oracle as O

    st, ua, va = make_case(n, 77 + n, u_scale=1.0)
    p = O.params(n, move)
    ref = O.advect(p, st)
    with sb.SoapFilm(sb.bubble(n, move), prec) as ctx:
        load(ctx, 0, st, ua, va)
        ctx.advect()
        for k in FIELDS:
            got = ctx.download(0, k + "_star")
            err = np.max(np.abs(got - ref[k])) / np.max(np.abs(ref[k]))
            print(f"  {prec} n={n} move={move} {k} {err:.2e}", flush=True)
            assert err <= TOL[prec], (k, err)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_advection_with_nan_samplers(prec):
    """A film with a NaN takes the NaN-skipping samplers everywhere: away from
    the NaN's neighbourhood the result is the one of the film without it."""
    n, m = 64, 128
    st, ua, va = make_case(n, 5, u_scale=1.0)
    out = []
    for nan in (False, True):
        s = {k: v.copy() for k, v in st.items()}
        if nan:
            s["eta"].reshape(n, m)[40, 100] = np.nan
        with sb.SoapFilm(sb.bubble(n, 0.01), prec) as ctx:
            load(ctx, 0, s, ua, va)
            ctx.advect()
            out.append({k: ctx.download(0, k + "_star") for k in FIELDS})
    for k in FIELDS:
        a, b = out
        assert np.max(np.abs(a[k] - b[k])[np.isfinite(b[k])] if k != "eta" else
                      np.abs(a[k] - b[k]).reshape(n, m)[:30]) <= TOL[prec] * np.max(np.abs(a[k]))
