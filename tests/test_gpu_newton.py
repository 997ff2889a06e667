"""QP Newton kernel at the edges of its storage rule and of its recurrences'
chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nen", [4, 5, 9, 10, 11, 66, 200, 1024, 1025, 3000])
def test_qp_newton_table_lengths(ngw_ctx, nen):
    """Both storage forms (tables in LDS up to 1024 points) and the chunk
    edges of the spline recurrences, against the oracle."""
    from oracle import oracle as O

    rng = np.random.default_rng(nen)
    nqp, width = 5, 20.0
    edft = rng.uniform(-15.0, 3.0, nqp)
    x = edft[None, :] - width / 2 + width / (nen - 1) * np.arange(nen)[:, None]
    pole = edft + rng.choice([-1.0, 1.0], nqp) * rng.uniform(15.0, 30.0, nqp)
    sig = np.asfortranarray(2.0 / (x - pole[None, :] + 1.5j))
    sigx = rng.uniform(-14.0, -8.0, nqp)
    vxc = sigx + rng.uniform(-1.0, 1.0, nqp)
    got = ngw_ctx.qp_newton(sig, width, edft, edft, sigx, vxc)
    for i in range(nqp):
        r = O.qp_solve(sig[:, i], width, edft[i], edft[i], sigx[i], vxc[i])
        for k in ("eqp", "zfac", "sigma0", "imsig"):
            assert abs(got[k][i] - r[k]) < 1e-9, (k, i)
        assert got["ierr"][i] == r["ierr"]
