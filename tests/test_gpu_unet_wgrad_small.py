"""Weight gradients over images smaller than a staged row of pixels (144) and just above
against the FP64 oracle (the bound of FP32 summation over the batch's pixels), and their
time against one image of as many pixels: many small images in a row once took six times
as long."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402
from oracle import unet_oracle as U  # noqa: E402

DEV = torch.device("cuda")


def _dev(x):
    return torch.from_numpy(U.to_bits(x).view(np.int16).copy()).to(DEV)


def _wgrad(d, x, C, N, H, W):
    part = torch.empty(_lib.fn("glide_unet_wgrad_chunks")(N, H, W) * 9 * C * C, device=DEV)
    dw = torch.empty(9 * C * C, device=DEV)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def go():
        _lib.call("glide_unet_conv3x3_wgrad", d.data_ptr(), C, x.data_ptr(), C, None, 0, N, H, W, part.data_ptr(),
                  dw.data_ptr(), st)

    go()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    for _ in range(10):
        go()
    b.record()
    torch.cuda.synchronize()
    return dw.cpu().numpy().reshape(9, C, C), a.elapsed_time(b)


@pytest.mark.parametrize("N,H,W", [(300, 1, 1), (150, 2, 1), (100, 1, 3), (40, 2, 2), (11, 5, 5), (7, 11, 13), (7, 12, 12),
                                   (7, 5, 29), (7, 16, 17)])
def test_small_images_match_oracle(N, H, W):
    C, P = 32, N * H * W
    rng = np.random.default_rng(P + W)
    x, dz = (U.bf16(rng.standard_normal((N, H, W, C)).astype(np.float32)) for _ in range(2))
    xd, dd = _dev(x), _dev(dz)
    got, t = _wgrad(dd, xd, C, N, H, W)
    ref, mag = U.conv3x3_wgrad(dz, x), U.conv3x3_wgrad(np.abs(dz), np.abs(x))
    assert np.all(np.abs(got - ref) <= (P + 2) * 2.0 ** -24 * mag)
    _, one = _wgrad(dd, xd, C, 1, 1, P)
    assert t < 2.5 * one, (t, one)
