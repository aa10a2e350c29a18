"""The row systems of the Gamma solve where a wave holds cells that are not
ordinary ones (needs an MI355X): broken cells at every place of a thread's
four (two) cells, on the phi seam and on both pole rows, concentrations above
the largest, and NaNs of the air, beside waves that have none of them. One
step without flow against the FP64 oracle, with the bounds that the
zero-thickness films of the parity tests have."""
import numpy as np
import pytest

import soapbubble_amd as sb
from cases import copy_state, load, make_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("where", ["inside", "seam", "north", "south"])
@pytest.mark.parametrize("n", [32, 101, 256])
def test_uncommon_cells(oracle, n, where, prec):
    print(f"uncommon cells {n} {where} {prec}", flush=True)
    m, dt = 2 * n, 0.003
    st, ua, va = make_case(n, 3)
    p = oracle.params(n, dt)
    with sb.SoapFilm(sb.bubble(n, dt), prec, tol=1e-12) as ctx:
        gmax = p.gamma_max
        row = {"inside": n // 3, "seam": n // 2, "north": 0, "south": n - 3}[where]
        col = np.arange(7 if where != "seam" else 11) + (9 if where != "seam" else m - 5)
        eta, gam = st["eta"].reshape(n, m), st["gamma"].reshape(n, m)
        for j in range(row, row + 3):
            eta[j, col % m] = 0.0
        # single cells: one at each place of a thread's cells
        for k in range(4):
            gam[(row + 1 + 2 * k) % n, (20 + 5 * k) % m] = 1.5 * gmax
        air = ua.reshape(-1)
        air[(row * m + np.array([1, 6, 30])) % air.size] = np.nan
        ref = copy_state(st)
        oracle.step(p, ref, ua, va, 1)
        load(ctx, 0, st, ua, va)
        ctx.step(1)
        got = ctx.state(0)
    tol = 1e-9 if prec == "fp64" else 1e-4
    for k in ("u_theta", "u_phi", "eta", "gamma"):
        ng, nr = np.isnan(got[k]), np.isnan(ref[k])
        both = ~(ng | nr)
        e = rel_l2(got[k][both], ref[k][both])
        print(f"  {k}: NaN {int(nr.sum())}, mismatched {int((ng != nr).sum())}, rel L2 {e:.2e}", flush=True)
        assert (ng != nr).sum() <= (0 if prec == "fp64" else 2), k
        assert e < tol, (k, e)
