"""V build: the parity transforms at the steps of their padding, on boxes and
supports of different length per axis, and the calls they leave to the FFT,
against the oracle's FFT Poisson solve."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

# FP64 transforms of a few hundred terms per axis: n eps log-like growth, far
# below this; M is a sum of ngrid products more.
TOL = 1e-12


def _case(extent, nfft, n_intp, seed, extra=()):
    rng = np.random.default_rng(seed)
    lo = [max(-m, -n // 2) for m, n in zip(extent, nfft)]
    hi = [min(m, n // 2 - 1) for m, n in zip(extent, nfft)]
    g = np.stack([rng.integers(a, b + 1, 400) for a, b in zip(lo, hi)], axis=1)
    g = np.unique(np.concatenate([g, [lo, hi, [0, 0, 0]]]), axis=0)
    g = np.concatenate([g, np.asarray(extra, g.dtype).reshape(-1, 3)]).astype(np.int32)
    zeta = np.asfortranarray(rng.normal(size=(len(g), n_intp)))
    return g, zeta


@pytest.mark.parametrize("extent,nfft", [
    ((15, 15, 15), (60, 60, 60)),     # m + 1 = 16: one tile of positions
    ((16, 16, 16), (62, 62, 62)),     # 17: two
    ((31, 31, 31), (126, 126, 126)),  # 32, h = 64: a full padding
    ((32, 32, 32), (130, 130, 130)),
    ((39, 39, 39), (158, 158, 158)),  # the 13 bohr molecule's box
    ((47, 47, 47), (190, 190, 190)),  # the largest extent of the kernels
    ((3, 14, 30), (24, 58, 120)),     # another length on every axis
    ((5, 5, 5), (10, 10, 10)),        # support as wide as the box: x = -n/2
    ((1, 0, 2), (2, 2, 4)),
    ((40, 10, 10), (250, 60, 60)),    # few positions, many frequencies
    ((50, 9, 9), (200, 40, 40)),      # beyond the kernels: FFT
    ((10, 10, 10), (260, 42, 42)),
])
def test_coulomb_kernel_boxes(ngw_ctx, extent, nfft):
    from oracle import oracle as O

    g, zeta = _case(extent, nfft, 5, sum(nfft))
    got = ngw_ctx.isdf_coulomb_kernel(zeta, g, nfft, 0.4, 9.0, 2.0)
    ref = O.isdf_kernel(zeta, g, nfft, 0.4, 9.0, 2.0)
    assert rel_err(got, ref) < TOL


@pytest.mark.parametrize("trunc", [0.0, 7.5])
@pytest.mark.parametrize("n_intp", [1, 63, 64, 65, 130])
def test_coulomb_kernel_columns_and_symmetry(ngw_ctx, n_intp, trunc):
    from oracle import oracle as O

    g, zeta = _case((9, 9, 9), (40, 40, 40), n_intp, n_intp)
    got = ngw_ctx.isdf_coulomb_kernel(zeta, g, (40, 40, 40), 0.5, trunc)
    ref = O.isdf_kernel(zeta, g, (40, 40, 40), 0.5, trunc)
    assert rel_err(got, ref) < TOL
    assert np.array_equal(got[:64, 64:], got[64:, :64].T)  # blocks off the diagonal tiles are mirrored


def test_coulomb_kernel_long_sum_and_leading_dimension(ngw_ctx):
    """k beyond one range of the symmetric product; M with a leading dimension
    of its own through the C entry."""
    import ctypes as C

    from nanogw_amd import _lib
    from oracle import oracle as O

    rng = np.random.default_rng(2)
    ax = np.arange(-9, 10)
    g = np.stack([a.ravel() for a in np.meshgrid(ax, ax, ax)], axis=1).astype(np.int32)
    zeta = np.asfortranarray(rng.normal(size=(len(g), 70)))
    ref = O.isdf_kernel(zeta, g, (40, 40, 40), 0.5, 8.0)
    out = np.full((77, 70), -1.0, order="F")
    dp, ip = C.POINTER(C.c_double), C.POINTER(C.c_int)
    nf = np.array([40, 40, 40], np.int32)
    _lib.check(_lib.load().ngw_isdf_coulomb_kernel(
        ngw_ctx.handle, len(g), 70, zeta.ctypes.data_as(dp), len(g), g.ctypes.data_as(ip), nf.ctypes.data_as(ip), 0.5,
        8.0, 1.0, out.ctypes.data_as(dp), 77), "ngw_isdf_coulomb_kernel")
    assert rel_err(out[:70], ref) < TOL
    assert np.all(out[70:] == -1.0)


def test_coincident_grid_points_go_to_the_fft(ngw_ctx):
    """A grid that names a point twice is accepted as before: both entries
    read the potential at the point."""
    from oracle import oracle as O

    g, zeta = _case((6, 6, 6), (24, 24, 24), 4, 3, extra=[[0, 0, 0]])
    zeta[np.all(g == 0, axis=1)] = zeta[-1]
    got = ngw_ctx.isdf_coulomb_kernel(zeta, g, (24, 24, 24), 0.5, 5.0)
    assert rel_err(got, O.isdf_kernel(zeta, g, (24, 24, 24), 0.5, 5.0)) < TOL


@pytest.mark.parametrize("extent,nfft,n_intp,head", [
    ((28, 28, 28), (114, 114, 114), 120, 20),   # batches of 35, 35, 35 and 15 columns
    ((28, 28, 28), (114, 114, 114), 77, 20),    # the last size of one batch
    ((39, 39, 39), (158, 158, 158), 35, 10),    # 32 and 3
])
def test_coulomb_kernel_batches(ngw_ctx, extent, nfft, n_intp, head):
    """Columns of the first and the last batch against calls of their own."""
    grid, zeta = _case(extent, nfft, n_intp, n_intp)
    m = ngw_ctx.isdf_coulomb_kernel(zeta, grid, nfft, 0.4, 7.5)
    for cols in (slice(0, head), slice(n_intp - head, n_intp)):
        part = ngw_ctx.isdf_coulomb_kernel(np.asfortranarray(zeta[:, cols]), grid, nfft, 0.4, 7.5)
        assert rel_err(m[cols, cols], part) < TOL


def test_coulomb_kernel_memory_of_many_columns(gpu, ngw_ctx):
    """12,000 columns: M on the device, V zeta, zeta and the transforms'
    intermediate, and no second array of M's order (half of M would be 0.6
    GB); M against the oracle on the first, last and middle columns."""
    import threading

    import torch

    from oracle import oracle as O

    n = 12000
    g, zeta = _case((4, 4, 4), (10, 10, 10), n, 7)
    ngw_ctx.isdf_coulomb_kernel(zeta[:, :64], g, (10, 10, 10), 0.4, 2.0)   # code objects loaded
    free = [torch.cuda.mem_get_info(0)[0]]
    done = threading.Event()

    def watch():
        while not done.wait(0.002):
            free.append(torch.cuda.mem_get_info(0)[0])

    t = threading.Thread(target=watch)
    t.start()
    try:
        m = ngw_ctx.isdf_coulomb_kernel(zeta, g, (10, 10, 10), 0.4, 2.0)
    finally:
        done.set()
        t.join()
    pick = np.r_[0:3, 6000:6003, n - 3:n]
    ref = O.isdf_kernel(np.asfortranarray(zeta[:, pick]), g, (10, 10, 10), 0.4, 2.0)
    assert rel_err(m[np.ix_(pick, pick)], ref) < TOL
    assert np.array_equal(m[:64, 64:], m[64:, :64].T)
    inter = 8 * 8 * 5 * 6 * 32 * min(n, 4096)                # 8 classes x (m + 1) x h x 32 frequencies a column
    need = 8 * (n * n + 2 * n * len(g)) + inter
    print("used", free[0] - min(free), "need", need)
    assert free[0] - min(free) < need + (128 << 20)
