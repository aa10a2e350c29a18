"""BIMOCQ next to the poles (needs an MI355X): a film that turns about the polar axis
as a rigid body carries a thickness that depends on theta alone into one that
does so again; what differs within a row is the rounding of the mapped
positions' theta."""
import numpy as np
import pytest

import soapbubble_amd as sb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turn", [0.1, 0.4])
def test_rows_stay_even(turn):
    """The thickness grows by one a row, so the differences are in cells: a theta
    within eight roundings of a unit vector (1.1e-16 each, 326 cells a radian)
    leaves 3e-13; one by the arc cosine of z next to the pole, where z hardly
    changes, leaves 1e-12 and more. Turned by less and by more than the quarter
    radian up to which the columns' angles are near (theta's always is)."""
    n, m = 1024, 2048
    th = (np.arange(n) + 0.5) * np.pi / n
    rows = lambda v: np.repeat(v, m)
    with sb.SoapFilm(sb.bubble(n, 1.0, airflow=False), "fp64", scalar_advection="bimocq") as ctx:
        ctx.upload(0, "u_theta", np.zeros((n - 1) * m))
        ctx.upload(0, "u_phi", rows(turn * np.sin(th)))
        ctx.upload(0, "eta", rows(np.arange(n) + 1.5))
        ctx.upload(0, "gamma", np.ones(n * m))
        ctx.advect()
        eta = ctx.download(0, "eta_star").reshape(n, m)
    spread = eta.max(axis=1) - eta.min(axis=1)
    print(f"  turned by {turn}: {spread[:16].max():.1e} in the northern rows, "
          f"{spread[-16:].max():.1e} in the southern", flush=True)
    assert spread[:16].max() < 3e-13, spread[:16]
    # (the southern rows' values, up to 1024, round by 1.1e-13 each)
    assert spread[-16:].max() < 3e-13 + 4 * 1.1e-13, spread[-16:]
