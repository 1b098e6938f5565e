"""The reference's example programs (saxpy, sgemv, 2-D stencil in five buffering styles)
on the wave64 DMA objects, through the C ABI, bit-exact against the CPU oracle."""
import numpy as np
import pytest

import cudadma_amd as cd
from cudadma_amd import examples as ex
from tests import oracle_lib as ol
from tests.oracle_lib import ptr

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    cd.lib()
    return torch.device("cuda:0")


def test_variant_tables(dev):
    assert ex.num_variants(ex.SAXPY) == 4 and ex.num_variants(ex.SGEMV) == 4 and ex.num_variants(ex.STENCIL2D) == 5
    assert "double buffer" in ex.variant_name(ex.STENCIL2D, 1)
    with pytest.raises(IndexError):
        ex.variant_name(ex.SAXPY, 4)


@pytest.mark.parametrize("variant", range(4))
@pytest.mark.parametrize("n", [1024, 3 * 1024, 1024 * 1031, 1 << 24])
def test_saxpy(dev, variant, n):
    O = ol.load()
    x, y = ol.uniform(n, 11), ol.uniform(n, 12)
    a = 0.8401877
    want = y.copy()
    O.oracle_saxpy(a, ptr(x), ptr(want), n)
    dx, dy = torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev)
    ex.saxpy(a, dx, dy, variant)
    torch.cuda.synchronize()
    assert np.array_equal(dy.cpu().numpy(), want)


def test_saxpy_ragged_and_empty(dev):
    O = ol.load()
    x, y = ol.uniform(1000, 13), ol.uniform(1000, 14)
    want = y.copy()
    O.oracle_saxpy(-1.5, ptr(x), ptr(want), 1000)
    dx, dy = torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev)
    ex.saxpy(-1.5, dx, dy, 0)                              # the baseline takes any length
    assert np.array_equal(dy.cpu().numpy(), want)
    with pytest.raises(cd.CudaDMAError, match="multiple of 1024"):
        ex.saxpy(1.0, dx, dy, 2)
    e = torch.empty(0, dtype=torch.float32, device=dev)
    ex.saxpy(1.0, e, e, 3)


@pytest.mark.parametrize("variant", range(4))
def test_sgemv_reference_driver_case(dev, variant):
    """A[j*n+i] = (i*j)%11, x[j] = j%11, alpha = 2 (sgemv_dma.cu:752-771): exact in any order.
    The reference runs n = m = 896; m is rounded to 1024 here so every variant's column multiple divides it."""
    n, m = 896, 1024
    i, j = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    a_int = (i * j) % 11
    x_int = np.arange(m) % 11
    a = torch.from_numpy(np.ascontiguousarray(a_int.T.astype(np.float32))).to(dev)     # (m, lda = n)
    x = torch.from_numpy(x_int.astype(np.float32)).to(dev)
    y = torch.full((n,), -1.0, dtype=torch.float32, device=dev)
    ex.sgemv(2.0, a, x, y, variant=variant)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().astype(np.int64), 2 * (a_int @ x_int))


@pytest.mark.parametrize("variant", range(4))
@pytest.mark.parametrize("n,m,lda", [(128, 512, 128), (200, 1024, 256), (1000, 1536, 1024), (4096, 4096, 4096)])
def test_sgemv_random(dev, variant, n, m, lda):
    O = ol.load()
    a = ol.uniform(m * lda, 21).reshape(m, lda)
    x = ol.uniform(m, 22)
    want = np.empty(n, dtype=np.float32)
    O.oracle_sgemv(n, m, 1.25, ptr(a), lda, ptr(x), ptr(want))
    da, dx = torch.from_numpy(a).to(dev), torch.from_numpy(x).to(dev)
    dy = torch.full((lda,), 3.0, dtype=torch.float32, device=dev)
    ex.sgemv(1.25, da, dx, dy, n=n, variant=variant)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    assert np.array_equal(got[:n], want)
    assert np.all(got[n:] == 3.0)                          # rows beyond n are not written


# the default variant's row tiles (16, 32, 64 and 128 rows by the number of workgroups) and panels: n around the lines between the
# tiles, m at one panel, between panels (the last one moves back) and below the smallest
@pytest.mark.parametrize("n", [1, 17, 4096, 4097, 8192, 8209, 16390, 28690])
@pytest.mark.parametrize("m", [32, 224, 256, 288, 480, 544, 768])
def test_sgemv_panels(dev, n, m):
    O = ol.load()
    lda = (n + 127) // 128 * 128
    a = ol.uniform(m * lda, 23).reshape(m, lda)
    x = ol.uniform(m, 24)
    want = np.empty(n, dtype=np.float32)
    O.oracle_sgemv(n, m, -0.75, ptr(a), lda, ptr(x), ptr(want))
    dy = torch.full((lda,), 3.0, dtype=torch.float32, device=dev)
    ex.sgemv(-0.75, torch.from_numpy(a).to(dev), torch.from_numpy(x).to(dev), dy, n=n)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    assert np.array_equal(got[:n], want)
    assert np.all(got[n:] == 3.0)


# the ring of stages: rows around the lines between its workgroups of 16, 32 and 64 rows, with and without a last stage that moves
# back, by one to three quarters, and one to six stages of the four; and what leaves it (fewer columns, more rows)
@pytest.mark.parametrize("n", [16, 4096, 4112, 8192, 8193, 10240, 10241, 16384, 16385])
@pytest.mark.parametrize("m", [96, 128, 160, 192, 352, 512, 640, 736])
def test_sgemv_ring(dev, n, m):
    O = ol.load()
    lda = (n + 127) // 128 * 128
    a = ol.uniform(m * lda, 27).reshape(m, lda)
    x = ol.uniform(m, 28)
    want = np.empty(n, dtype=np.float32)
    O.oracle_sgemv(n, m, 0.5, ptr(a), lda, ptr(x), ptr(want))
    dy = torch.full((lda,), 3.0, dtype=torch.float32, device=dev)
    ex.sgemv(0.5, torch.from_numpy(a).to(dev), torch.from_numpy(x).to(dev), dy, n=n)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    assert np.array_equal(got[:n], want)
    assert np.all(got[n:] == 3.0)


def test_sgemv_special_values(dev):
    """Infinities and NaN stay in their rows (lanes that sum other columns of the same rows meanwhile see them too), zeros keep
    their sign through alpha, and denormal products count."""
    n, m = 48, 416
    O = ol.load()
    a = ol.uniform(m * 128, 29).reshape(m, 128)
    x = ol.uniform(m, 30)
    a[[0, 33, 70, 127, 128, 300, 415], [1, 2, 3, 4, 5, 6, 7]] = [np.inf, -np.inf, np.nan, np.inf, np.nan, -np.inf, np.inf]
    a[40, 1] = -np.sign(x[40] * x[0]) * np.inf              # inf - inf
    a[:, 8] = 0.0
    a[:, 9] *= np.float32(2.0 ** -126)
    a[:, 10] = -0.0
    want = np.empty(n, dtype=np.float32)
    O.oracle_sgemv(n, m, -1.0, ptr(a), 128, ptr(x), ptr(want))
    dy = torch.zeros(128, dtype=torch.float32, device=dev)
    ex.sgemv(-1.0, torch.from_numpy(a).to(dev), torch.from_numpy(x).to(dev), dy, n=n)
    got = dy.cpu().numpy()[:n]
    nan = np.isnan(want)
    assert nan.sum() >= 3 and np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


# a leading dimension far beyond what n needs: the columns of one panel lie more than 2 GiB apart (256, 128 and 32 columns)
@pytest.mark.parametrize("n,m,lda,variant", [(16, 256, 2_200_064, 3), (4160, 288, 2_200_064, 3), (8200, 288, 4_300_032, 3), (40, 32, 17_400_064, 3),
                                             (40, 32, 17_400_064, 2), (40, 256, 17_400_064, 3), (40, 128, 67_108_860, 3), (40, 128, 67_108_864, 3)])
def test_sgemv_columns_far_apart(dev, n, m, lda, variant):
    O = ol.load()
    pad = (n + 127) // 128 * 128
    a = ol.uniform(m * pad, 25).reshape(m, pad)
    x = ol.uniform(m, 26)
    want = np.empty(n, dtype=np.float32)
    O.oracle_sgemv(n, m, 1.5, ptr(a), pad, ptr(x), ptr(want))
    da = torch.empty((m, lda), dtype=torch.float32, device=dev)        # only the rows that are read are filled
    da[:, :pad] = torch.from_numpy(a).to(dev)
    dy = torch.full((pad,), 3.0, dtype=torch.float32, device=dev)
    ex.sgemv(1.5, da, torch.from_numpy(x).to(dev), dy, n=n, variant=variant)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    assert np.array_equal(got[:n], want) and np.all(got[n:] == 3.0)


def test_sgemv_argument_checks(dev):
    a = torch.zeros((96, 128), dtype=torch.float32, device=dev)
    x = torch.zeros(96, dtype=torch.float32, device=dev)
    y = torch.zeros(128, dtype=torch.float32, device=dev)
    with pytest.raises(cd.CudaDMAError, match="multiple of 256"):
        ex.sgemv(1.0, a, x, y, variant=0)
    a2 = torch.zeros((64, 100), dtype=torch.float32, device=dev)
    with pytest.raises(cd.CudaDMAError, match="must cover 128 rows"):
        ex.sgemv(1.0, a2, torch.zeros(64, dtype=torch.float32, device=dev), y, variant=2)


@pytest.mark.parametrize("variant", range(5))
@pytest.mark.parametrize("full_cross", [False, True])
@pytest.mark.parametrize("dims", [(32, 4, 2), (96, 20, 6), (960, 160, 8)])
def test_stencil2d(dev, variant, full_cross, dims):
    """Reference geometry (params_directed.h: 960 x 160 tiles of 32 x 4, radius 4) at a few depths."""
    O = ol.load()
    dimx, dimy, dimz = dims
    r = ex.STENCIL2D_RADIUS
    shape = (dimz + 2 * r, dimy + 2 * r, dimx + 2 * r, 2)
    src = ol.uniform(int(np.prod(shape)), 31)
    want = np.full(src.size, -7.0, dtype=np.float32)
    O.oracle_stencil2d(ptr(src), ptr(want), dimx, dimy, dimz, r, r if full_cross else r - 1)
    dsrc = torch.from_numpy(src).to(dev).view(shape)
    ddst = torch.full(shape, -7.0, dtype=torch.float32, device=dev)
    ex.stencil2d(dsrc, ddst, variant, full_cross)
    torch.cuda.synchronize()
    assert np.array_equal(ddst.cpu().numpy().ravel(), want)


# every tile shape, and dimensions that the tile does not divide (its last tile moves back to fit): 32 x 4 below 64 columns or 8
# rows, 64 x 8 above, 64 x 32 where the volume exceeds the caches
@pytest.mark.parametrize("variant", range(5))
@pytest.mark.parametrize("full_cross", [False, True])
@pytest.mark.parametrize("dims", [(32, 20, 2), (96, 4, 6), (64, 8, 2), (96, 12, 4), (160, 36, 6), (64, 44, 130), (288, 60, 740)])
def test_stencil2d_tile_shapes(dev, variant, full_cross, dims):
    O = ol.load()
    dimx, dimy, dimz = dims
    r = ex.STENCIL2D_RADIUS
    shape = (dimz + 2 * r, dimy + 2 * r, dimx + 2 * r, 2)
    src = ol.uniform(int(np.prod(shape)), 33)
    want = np.full(src.size, -7.0, dtype=np.float32)
    O.oracle_stencil2d(ptr(src), ptr(want), dimx, dimy, dimz, r, r if full_cross else r - 1)
    dsrc = torch.from_numpy(src).to(dev).view(shape)
    buf = torch.full((src.size + 2,), -7.0, dtype=torch.float32, device=dev)
    for first in (0, 2):                                   # a destination that is 16-byte aligned, and one that is 8-byte aligned
        ddst = buf[first:first + src.size].view(shape)
        ex.stencil2d(dsrc, ddst, variant, full_cross)
        torch.cuda.synchronize()
        assert np.array_equal(ddst.cpu().numpy().ravel(), want)
        buf.fill_(-7.0)


def test_stencil2d_argument_checks(dev):
    r = ex.STENCIL2D_RADIUS
    odd = torch.zeros((3 + 2 * r, 4 + 2 * r, 32 + 2 * r, 2), dtype=torch.float32, device=dev)
    with pytest.raises(cd.CudaDMAError, match="must be even"):
        ex.stencil2d(odd, odd.clone(), 1)
    ex.stencil2d(odd, odd.clone(), 0)                      # one buffer: any depth
    bad = torch.zeros((2 + 2 * r, 5 + 2 * r, 32 + 2 * r, 2), dtype=torch.float32, device=dev)
    with pytest.raises(cd.CudaDMAError, match="multiple of"):
        ex.stencil2d(bad, bad.clone(), 0)
