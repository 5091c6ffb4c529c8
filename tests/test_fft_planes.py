"""The fused z/y plane pass: the configuration a convolution reports."""
import pytest

from mini_mdft_amd import FP32, FP64, luc
from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _conv(n, prec):
    shape, L = (2, n, n), (2.0, 0.3 * n, 0.3 * n)
    g, ag = M.SpatialGrid(shape, L), M.AngularGrid(1, 1)
    tab = luc.synthetic_c(1, 1, luc.nq_for(luc.qmax_of_grid(shape, L), luc.DQ_TIP3P), seed=3)
    return shape, ag, M.Convolution.from_table(tab, g, ag, M.OrientationProjectionMap(ag), prec)


@pytest.mark.parametrize("prec", [FP32, FP64])
@pytest.mark.parametrize("n", [12, 20, 28, 36, 72])
def test_reported_threads(n, prec):
    """Planes compiled with one thread count (256 up to 32, else 512) report it,
    before and after tuning."""
    shape, ag, conv = _conv(n, prec)
    p = torch.zeros((ag.m_np,) + shape, dtype=torch.complex64 if prec == FP32 else torch.complex128, device="cuda")
    for _ in range(2):
        c = conv.fft_config()
        if c["plane"]:
            assert c["plane_threads"] == (256 if n <= 32 else 512)
        conv.execute(p)


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n", [14, 49, 77, 81, 96, 100, 128])
def test_forced(n, dtype):
    """Planes in LDS once or twice, with radices above 5, with 256 and 512 threads
    asked for: bitwise the axis passes."""
    if dtype == torch.complex128 and n > 100:  # one plane does not fit in LDS
        with pytest.raises(M.MDFTError, match="does not apply"):
            M.fft3d_config(torch.zeros((1, 1, n, n), dtype=dtype, device="cuda"), -1, True)
        return
    x = torch.randn((2, 2, n, n), dtype=dtype, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    for sign in (-1, 1):
        ref = x.clone()
        M.fft3d_config(ref, sign, False, wz=3, wy=3)
        for threads in (256, 512):
            y = x.clone()
            M.fft3d_config(y, sign, True, threads)
            assert torch.equal(y, ref), threads


@pytest.mark.parametrize("shape", [(1, 2, 130, 130), (1, 2, 49, 50), (1, 2, 1, 8)])
def test_refused(shape):
    """Too large for LDS, unequal sides with a radix above 5, and no y axis."""
    with pytest.raises(M.MDFTError, match="does not apply"):
        M.fft3d_config(torch.zeros(shape, dtype=torch.complex64, device="cuda"), -1, True)


@pytest.mark.parametrize("prec", [FP32, FP64])
@pytest.mark.parametrize("n", [49, 64, 81, 96])
def test_reported_configuration_is_accepted(n, prec):
    """What a tuned convolution reports runs as mdft_fft3d_config."""
    shape, ag, conv = _conv(n, prec)
    dtype = torch.complex64 if prec == FP32 else torch.complex128
    x = torch.randn((ag.m_np,) + shape, dtype=dtype, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    conv.execute(x.clone())
    c = conv.fft_config()
    assert c.pop("tuned")
    y, ref = x.clone(), x.clone()
    M.fft3d_config(y, -1, bool(c.pop("plane")), **c)
    M.fft3d(ref, -1)
    assert torch.equal(y, ref)


@pytest.mark.parametrize("n", [64, 96, 100])
@pytest.mark.parametrize("dt", [0, 1])
def test_no_transforms(n, dt):
    """A batch of none is done, in planes as in axis passes."""
    from mini_mdft_amd._lib import check, lib

    x = torch.zeros(1, dtype=torch.complex128, device="cuda")
    check(lib().mdft_fft3d(x.data_ptr(), 0, 2, n, n, -1, dt, None))
