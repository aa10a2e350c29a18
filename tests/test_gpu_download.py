"""Fields uploaded and downloaded again, bit for bit (needs an MI355X): sizes on
either side of the staging buffer and of the cut into several threads."""
import numpy as np
import pytest

import soapbubble_amd as sb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [4, 101, 512, 725, 1024, 1450])
def test_round_trip(prec, n):
    rng = np.random.default_rng(n)
    with sb.SoapFilm(sb.bubble(n, 0.001), prec) as ctx:
        for field, rows in (("eta", n), ("u_theta", n - 1)):
            a = rng.uniform(0.5, 1.5, rows * 2 * n)
            if prec == "mixed":
                a = a.astype(np.float32).astype(np.float64)
            ctx.upload(0, field, a)
            assert np.array_equal(ctx.download(0, field), a), (prec, n, field)
