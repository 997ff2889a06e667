"""FP64 operator kernels at the edges of their dispatch rules: every K1 / K2 /
K3 tile form with remainders in each dimension, and the one-vector kernels
over the nv steps of their column chunks."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

# Sums of at most 1e5 terms with random signs in FP64: sqrt(n) eps = 4e-14
# times a cancellation of the result against its terms of at most ten.
TOL = 1e-12


def _system(nmu, nv, nc, seed):
    rng = np.random.default_rng(seed)
    psi = np.asfortranarray(rng.normal(size=(nmu, nv + nc)) / np.sqrt(nmu))
    g = rng.normal(size=(nmu, max(4, nmu // 2)))
    m = np.asfortranarray(g @ g.T / nmu)
    e = np.concatenate([np.sort(rng.uniform(-1.8, -0.5, nv)), np.sort(rng.uniform(-0.3, 4.0, nc))])
    return psi, m, e


def _operator(psi, m, e, nv, x, tda):
    """y (ncv, B) of the factored operator, FP64."""
    nc = psi.shape[1] - nv
    r = (e[nv:, None] - e[None, :nv]).reshape(-1)
    s = np.ones_like(r) if tda else np.sqrt(r)
    y = np.empty_like(x)
    for b in range(x.shape[1]):
        xb = (s * x[:, b]).reshape(nc, nv)
        u = m @ ((psi[:, nv:] @ xb) * psi[:, :nv]).sum(axis=1)
        g = (psi[:, nv:].T @ (psi[:, :nv] * u[:, None])).reshape(-1)
        y[:, b] = r * x[:, b] + 2.0 * g if tda else r * r * x[:, b] + 4.0 * s * g
    return y


def _check(ctx, nmu, nv, nc, blksz, tda=False):
    psi, m, e = _system(nmu, nv, nc, 7 * nmu + nv)
    x = np.random.default_rng(blksz).normal(size=(nv * nc, blksz))
    ctx.set_isdf(psi, m, e, nv)
    ctx.set_precision("f64")
    y = ctx.matvec_isdf_BLOCK(x, tamm_d=tda)
    pick = np.unique(np.concatenate([np.arange(min(blksz, 40)), np.arange(max(0, blksz - 40), blksz)]))
    ref = _operator(psi, m, e, nv, x[:, pick], tda)
    assert rel_err(y[:, pick], ref) < TOL
    return y


@pytest.mark.parametrize("nmu,nv,nc,blksz", [
    (33, 5, 17, 3),       # 16-row K1, 16 x 16 K2 and K3 waves, remainders everywhere
    (16, 2, 16, 8),       # no remainder
    (15, 1, 15, 2),       # less than one block of k
    (40, 70, 20, 3),      # nv > 64: slots summed by their own kernel
    (50, 64, 18, 2),      # nv = one K1 tile: one or two slots per vector
    (50, 65, 18, 2),
    (301, 9, 31, 101),    # 32-row K1
    (400, 25, 37, 100),   # 64 x 64 K1, 32 x 32 K2
    (100, 24, 250, 80),   # 32 x 16 K3 waves
    (90, 47, 129, 85),    # 64 x 64 K3
    (130, 33, 200, 160),  # 128 x 64 K3
    (520, 3, 1030, 3900), # 128-row K1, 128 x 64 K2
])
def test_block_operator_tile_forms(ngw_ctx, nmu, nv, nc, blksz):
    _check(ngw_ctx, nmu, nv, nc, blksz)


@pytest.mark.parametrize("tda", [False, True])
@pytest.mark.parametrize("nmu,nv,nc", [
    (1, 1, 1), (1, 20, 3), (2, 17, 5), (31, 1, 40), (480, 8, 56), (67, 15, 33), (64, 16, 32), (65, 17, 31),
    (99, 32, 70), (101, 33, 71), (129, 64, 66), (131, 65, 67), (961, 48, 300), (203, 113, 257), (2777, 101, 901)])
def test_one_vector_operator_forms(ngw_ctx, nmu, nv, nc, tda):
    _check(ngw_ctx, nmu, nv, nc, 1, tda)


def test_block_size_does_not_change_a_column(ngw_ctx):
    """The FP64 tile forms add every sum in the same order, so a column has
    the same bits in calls of any width."""
    nmu, nv, nc = 300, 13, 90
    wide = _check(ngw_ctx, nmu, nv, nc, 700)
    x = np.random.default_rng(700).normal(size=(nv * nc, 700))
    for n in (2, 30, 333):
        assert np.array_equal(ngw_ctx.matvec_isdf_BLOCK(x[:, :n]), wide[:, :n]), n


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (63, 65, 15), (64, 64, 16), (65, 129, 17),   # 64 x 64 tiles
    (1000, 1910, 33), (1023, 2049, 40),                     # 240 wide tiles: 64 x 64; 272: 64 x 128
    (2049, 1025, 18)])
def test_plain_gemm_tile_forms(gpu, ngw_ctx, m, n, k):
    import torch

    g = torch.Generator(device="cuda").manual_seed(m)
    a = torch.randn(k, m, generator=g, device="cuda", dtype=torch.float64)   # column-major (m, k)
    b = torch.randn(n, k, generator=g, device="cuda", dtype=torch.float64)
    c = torch.full((n, m), float("nan"), device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    ngw_ctx.gemm_f64_dev(m, n, k, a.data_ptr(), m, b.data_ptr(), k, c.data_ptr(), m)
    ngw_ctx.synchronize()
    ref = b.cpu().numpy() @ a.cpu().numpy()
    assert rel_err(c.cpu().numpy(), ref) < TOL
