"""Low-precision operator with M-tile counts on both sides of every division
of the XCDs into M groups (1 to 9 tiles and more, with remainders)."""
import numpy as np
import pytest

from test_gpu_f64_tiles import _operator, _system

pytestmark = pytest.mark.gpu

# Per unit of the largest element: the operands' rounding (2^-8, 2^-11, 2^-16;
# for FP32 that of sums of up to 2^11 terms with random signs, 2^-24 x 2^5.5),
# sixteen times for the three chained products and their largest partial sums.
TOL = {"bf16": 16 * 2.0**-8, "f16": 16 * 2.0**-11, "bf16x3": 16 * 2.0**-16, "f32": 16 * 2.0**-18}


@pytest.mark.parametrize("prec", ["f32", "bf16", "bf16x3", "f16"])
@pytest.mark.parametrize("nmu,nc,nv,blksz", [
    (40, 100, 3, 5),       # one M tile in K1 and K3, fewer N tiles than XCDs
    (129, 256, 9, 60),     # 2 and 2
    (384, 257, 17, 30),    # 3 and 3
    (500, 640, 31, 37),    # 4 and 5
    (700, 900, 12, 90),    # 6 and 8
    (1000, 1025, 7, 111),  # 8 and 9
    (2050, 1200, 5, 64),   # 17 and 10
])
def test_every_tile_is_computed_once(ngw_ctx, prec, nmu, nc, nv, blksz):
    psi, m, e = _system(nmu, nv, nc, nmu + nc)
    m *= nmu  # the product comparable with the diagonal
    x = np.random.default_rng(blksz).normal(size=(nv * nc, blksz))
    ngw_ctx.set_isdf(psi, m, e, nv)
    ngw_ctx.set_precision(prec)
    try:
        y = ngw_ctx.matvec_isdf_BLOCK(x, tamm_d=True)
    finally:
        ngw_ctx.set_precision("f64")
    # the operator's product alone: the diagonal would hide a small error
    d = ((e[nv:, None] - e[None, :nv]).reshape(-1))[:, None] * x
    ref = _operator(psi, m, e, nv, x, True) - d
    assert np.abs(y - d - ref).max() < TOL[prec] * np.abs(ref).max()


@pytest.mark.parametrize("nmu,nc,nv,blksz", [
    (1100, 1030, 33, 500),   # wide K1 and K3 tiles, remainders in M and N
    (1100, 700, 20, 1000),   # k of K1 too short, K3 wide
    (900, 1281, 129, 117),   # K1 wide (an odd nv above one slot), k of K3 too short
])
def test_wide_tiles_do_not_change_a_column(ngw_ctx, nmu, nc, nv, blksz):
    """Large FP16 calls take 256-column tiles: the bits of a column are those
    of a narrow call, which takes the 128-column ones."""
    psi, m, e = _system(nmu, nv, nc, nmu + nc)
    m *= nmu
    x = np.random.default_rng(blksz).normal(size=(nv * nc, blksz))
    ngw_ctx.set_isdf(psi, m, e, nv)
    ngw_ctx.set_precision("f16")
    try:
        wide = ngw_ctx.matvec_isdf_BLOCK(x)
        narrow = ngw_ctx.matvec_isdf_BLOCK(x[:, :9])
    finally:
        ngw_ctx.set_precision("f64")
    assert np.array_equal(wide[:, :9], narrow)
    d = ((e[nv:, None] - e[None, :nv]).reshape(-1) ** 2)[:, None] * x[:, -12:]
    ref = _operator(psi, m, e, nv, x[:, -12:], False) - d
    assert np.abs(wide[:, -12:] - d - ref).max() < TOL["f16"] * np.abs(ref).max()
