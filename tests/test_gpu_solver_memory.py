"""Solver parts that are allocated when a film first needs them, where the memory
for them is missing (needs an MI355X; SF_FAIL_ALLOC, a test hook, fails the named
part after its last array): without the spectral preconditioner's arrays
multigrid takes the film, without either the step reports the error, each
time it is called."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import copy_state, load, make_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu

FIELDS = ("u_theta", "u_phi", "eta", "gamma")
RADIUS = 0.05
# as the stiff films' comparison with the oracle: FP32 fields (6e-8) over a few
# steps, u by the gradient of an FP32 Gamma
TOL = 5e-6


@pytest.mark.parametrize("part", ["coefficients", "spectral"])
@pytest.mark.parametrize("graph", [True, False])
def test_multigrid_takes_over(graph, part, monkeypatch, capfd):
    from oracle import oracle as O

    n, dt = 64, 0.02
    st, ua, va = make_case(n, 95, u_scale=0.1)
    monkeypatch.setenv("SF_FAIL_ALLOC", part)
    monkeypatch.setenv("SF_SOLVE_TRACE", "1")
    with sb.SoapFilm(sb.bubble(n, dt, radius=RADIUS), "mixed", use_graph=graph) as ctx:
        load(ctx, 0, st, ua, va)
        ctx.step(4)
        ctx.step(5)
        got, s = ctx.state(0), ctx.stats(0)
    err = capfd.readouterr().err
    assert "multigrid from here on" in err and "spectral preconditioner" not in err
    assert s["failed_solves"] == 0, s
    ref = copy_state(st)
    O.step(O.params(n, dt, radius=RADIUS), ref, ua, va, 9)
    for k in FIELDS:
        assert rel_l2(got[k], ref[k]) < TOL, (k, rel_l2(got[k], ref[k]))


@pytest.mark.parametrize("method", ["auto", "mg"])
def test_no_memory_for_either(method, monkeypatch):
    n, dt = 64, 0.02
    st, ua, va = make_case(n, 95, u_scale=0.1)
    monkeypatch.setenv("SF_FAIL_ALLOC", "spectral,multigrid")
    if method == "mg":
        with pytest.raises(sb.SoapFilmError) as e:
            sb.SoapFilm(sb.bubble(n, dt, radius=RADIUS), "mixed", inner_method=method)
        assert e.value.code == 4
        return
    with sb.SoapFilm(sb.bubble(n, dt, radius=RADIUS), "mixed", use_graph=True) as ctx:
        load(ctx, 0, st, ua, va)
        for _ in range(3):
            with pytest.raises(sb.SoapFilmError) as e:
                ctx.step(3)
            assert e.value.code == 4
        assert np.isfinite(ctx.download(0, "eta")).all()
