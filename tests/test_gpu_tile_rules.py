"""Dispatch rules of the operator kernels at the sizes where they change over."""
import numpy as np
import pytest

from conftest import rel_err
from nanogw_amd.lanczos import IsdfContext
from test_gpu_f64_tiles import TOL, _operator, _system
from test_gpu_lowp_tiles import TOL as LOWP_TOL

pytestmark = pytest.mark.gpu


def test_a_chosen_tile_configuration_is_used_as_given(gpu):
    """Every index names one tile at every launch width; only while none was
    set or tuned does the size decide."""
    nmu, nv, nc, wide = 1100, 33, 1030, 500   # 9 x 65 tiles of 128 x 256 in K1 and K3, k 1056 and 1120
    with IsdfContext(0) as ctx:
        ctx.set_isdf(*_system(nmu, nv, nc, 3), nv)
        assert ctx.tile_config(wide) == (0, 0)   # FP64
        for prec in ("f32", "bf16", "bf16x3", "f16"):
            ctx.set_precision(prec)
            assert ctx.tile_config(9) == (0, 0)
            assert ctx.tile_config(wide) == ((4, 5) if prec == "f16" else (0, 0))
            chosen = ctx.autotune(wide, reps=1)
            assert ctx.tile_config(wide) == ctx.tile_config(9) == chosen
            for c in range(6):
                ctx.set_tile_config(c, 5 - c)
                assert ctx.tile_config(wide) == ctx.tile_config(9) == (c, 5 - c)


def test_more_columns_than_a_grid_of_narrow_tiles(gpu):
    """K1 over more 64 x 64 tiles than one launch has threads for (2^32):
    4096 points and 131,075 vectors of 128 valence states."""
    import torch

    nmu, nv, nc, b = 4096, 128, 1, 131075
    psi, m, e = _system(nmu, nv, nc, 5)
    x = torch.randn(b, nv * nc, device="cuda", dtype=torch.float64, generator=torch.Generator(device="cuda").manual_seed(1))
    y = torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    with IsdfContext(0) as ctx:   # 22 GB of work arrays, freed with it
        ctx.set_isdf(psi, m, e, nv)
        ctx.matvec_dev(x.data_ptr(), y.data_ptr(), nv * nc, b)
        ctx.synchronize()
    assert not torch.isnan(y).any()
    pick = np.r_[0:4, 65534:65540, b - 4:b]
    ref = _operator(psi, m, e, nv, np.ascontiguousarray(x[pick].cpu().numpy().T), False)
    assert rel_err(y[pick].cpu().numpy().T, ref) < TOL


@pytest.mark.parametrize("prec", ["f32", "bf16", "bf16x3", "f16"])
@pytest.mark.parametrize("nv", [3, 4])   # K3's element-wise and 16-byte epilogues
@pytest.mark.parametrize("nc", [1, 8, 15, 16, 17, 63, 65, 72, 80, 129])
def test_k3_tiles_mostly_past_the_end(ngw_ctx, prec, nv, nc):
    """K3 tiles of 128 rows with all but a few past nc: what the epilogue
    skips and what it writes meet at every group and batch of rows."""
    nmu, b = 60, 23
    psi, m, e = _system(nmu, nv, nc, nc)
    m *= nmu
    x = np.random.default_rng(nv).normal(size=(nv * nc, b))
    ngw_ctx.set_isdf(psi, m, e, nv)
    ngw_ctx.set_precision(prec)
    try:
        y = ngw_ctx.matvec_isdf_BLOCK(x, tamm_d=True)
    finally:
        ngw_ctx.set_precision("f64")
    d = ((e[nv:, None] - e[None, :nv]).reshape(-1))[:, None] * x
    ref = _operator(psi, m, e, nv, x, True) - d
    assert np.abs(y - d - ref).max() < LOWP_TOL[prec] * np.abs(ref).max()


@pytest.mark.parametrize("nmu,nc,nv,blksz,tiles", [
    (1100, 1030, 33, 500, (4, 5)),   # 9 x 65 tiles of 128 x 256 in K1 and K3, remainders in M and N
    (1100, 1030, 32, 520, (4, 5)),   # K3's 16-byte epilogue
    (1100, 700, 20, 1100, (0, 5)),   # k of K1 704; 6 x 86 tiles in K3, 16-byte epilogue
    (900, 1281, 129, 130, (4, 0)),   # 8 x 66 tiles in K1, vectors of two partial sums; k of K3 960
    (600, 1030, 300, 90, (4, 0)),    # 5 x 106 tiles in K1, vectors of three and four partial sums
    (1100, 1030, 33, 400, (0, 0)),   # 9 x 52
])
def test_wide_fp16_tiles_keep_the_bits_of_the_narrow_ones(gpu, nmu, nc, nv, blksz, tiles):
    """The tiles the size rule takes for large FP16 launches, against the
    128 x 128 ones on the same call and on its first columns alone (a column's
    place decides where K1's partial sums are cut, so only leading columns keep
    their bits)."""
    psi, m, e = _system(nmu, nv, nc, nmu + nc)
    m *= nmu
    x = np.random.default_rng(blksz).normal(size=(nv * nc, blksz))
    with IsdfContext(0) as ctx:
        ctx.set_isdf(psi, m, e, nv)
        ctx.set_precision("f16")
        assert ctx.tile_config(blksz) == tiles
        assert ctx.tile_config(9) == (0, 0)
        wide = ctx.matvec_isdf_BLOCK(x)
        few = ctx.matvec_isdf_BLOCK(x[:, :9])
        ctx.set_tile_config(0, 0)
        assert ctx.tile_config(blksz) == (0, 0)
        narrow = ctx.matvec_isdf_BLOCK(x)
    assert np.array_equal(wide, narrow)
    assert np.array_equal(wide[:, :9], few)
    d = ((e[nv:, None] - e[None, :nv]).reshape(-1) ** 2)[:, None] * x[:, -6:]
    ref = _operator(psi, m, e, nv, x[:, -6:], False) - d
    assert np.abs(wide[:, -6:] - d - ref).max() < LOWP_TOL["f16"] * np.abs(ref).max()


@pytest.mark.parametrize("nmu,nv,nc,blksz", [
    (401, 25, 37, 700),    # 26 x 44 K2 tiles of 16 x 16, more than a wave per SIMD: 13 x 22 of 32 x 32
    (515, 1, 20, 601),     # 33 x 38, and K1 without LDS: K2 adds the two slots of a vector
    (515, 2, 70, 299),     # 33 x 19 = 627: 16 x 16 waves, adding the slots
    (2048, 1, 18, 1025),   # 64 x 33 = 2112 tiles of 32 x 32: 128 x 64
])
def test_f64_k2_forms(ngw_ctx, nmu, nv, nc, blksz):
    """K2's 32 x 32 LDS tiles and the sizes beside them.  Leading columns have
    the same bits in calls of every width from two on; one vector alone takes
    kernels that split its sums, and agrees to rounding."""
    psi, m, e = _system(nmu, nv, nc, nmu)
    x = np.random.default_rng(nmu).normal(size=(nv * nc, blksz))
    ngw_ctx.set_isdf(psi, m, e, nv)
    ngw_ctx.set_precision("f64")
    y = ngw_ctx.matvec_isdf_BLOCK(x)
    pick = np.r_[0:20, blksz // 2:blksz // 2 + 20, blksz - 20:blksz]
    assert rel_err(y[:, pick], _operator(psi, m, e, nv, x[:, pick], False)) < TOL
    for n in (2, 35, 261):
        assert np.array_equal(ngw_ctx.matvec_isdf_BLOCK(x[:, :n]), y[:, :n]), n
    one = ngw_ctx.matvec_isdf_BLOCK(x[:, :1])
    assert rel_err(one, y[:, :1]) < TOL
