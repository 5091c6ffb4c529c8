"""The FFT's per-axis tiles: every compiled width against tiles of the run-time
kernels (3 lines) bit for bit, on whole and ragged tiles of lines and of columns
and on strides below a tile."""
import numpy as np
import pytest

from mini_mdft_amd import mdft as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# whole tiles of z lines (16 x 16 of 64), ragged ones, strides of 2 to 8, 27 and 63 columns
SHAPES = [(1, 16, 16, 64), (2, 64, 5, 4), (1, 100, 2, 3), (1, 128, 1, 5), (1, 91, 1, 7), (3, 8, 9, 63), (1, 32, 7, 27),
          (1, 66, 1, 2), (2, 12, 65, 8)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
def test_widths(shape, dtype):
    r = np.random.default_rng(5)
    x = torch.from_numpy(r.standard_normal(shape) + 1j * r.standard_normal(shape)).to(dtype).cuda()
    ref = x.clone()
    M.fft3d_config(ref, -1, False, wz=3, wy=3, wx=3)
    for w in (0, 4, 5, 7, 8, 11, 16, 32, 64):  # contiguous tiles of 512 or 1024 values are among them
        y = x.clone()
        M.fft3d_config(y, -1, False, wz=w, wy=w, wx=w)
        assert torch.equal(y, ref), w
    y = x.clone()
    M.fft3d(y, -1)
    assert torch.equal(y, ref)
