"""The convolution's weight gradient against the float64 oracle where its
tiling can go wrong: images narrower than a fragment's 8 pixels, widths that
are not multiples of 8, several images, chunk remainders, and every 32-channel
group of both inputs.

Tolerance per entry: an FP32 sum of P products in any order is off by at most
(P + 2) 2^-24 times the sum of the products' magnitudes.  The bias gradient of
the same launch equals glide_unet_bias_grad's bit for bit."""
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


@pytest.mark.parametrize("N,H,W", [(1, 1, 1), (1, 3, 5), (5, 2, 3), (2, 5, 8), (1, 16, 24), (3, 33, 40), (1, 70, 61),
                                   (2, 48, 64)])
@pytest.mark.parametrize("CA,CB,Co", [(32, 0, 32), (64, 32, 96)])
def test_wgrad_matches_oracle(N, H, W, CA, CB, Co):
    rng = np.random.default_rng(H * W + CA)
    mk = lambda c: U.bf16(rng.standard_normal((N, H, W, c)).astype(np.float32))   # noqa: E731
    xa, xb, dz = mk(CA), mk(max(CB, 1))[..., :CB], mk(Co)
    Ci, P = CA + CB, N * H * W
    part = torch.empty(_lib.fn("glide_unet_wgrad_chunks")(N, H, W) * 9 * Co * Ci, device=DEV)
    dw = torch.empty(9 * Co * Ci, device=DEV)
    a, b, d = _dev(xa), (_dev(xb) if CB else None), _dev(dz)
    _lib.call("glide_unet_conv3x3_wgrad", d.data_ptr(), Co, a.data_ptr(), CA, b.data_ptr() if CB else None, CB, N, H,
              W, part.data_ptr(), dw.data_ptr(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    part2 = torch.empty(part.numel() + _lib.fn("glide_unet_wgrad_chunks")(N, H, W) * Co, device=DEV)
    dw2, db, db2 = torch.empty_like(dw), torch.empty(Co, device=DEV), torch.empty(Co, device=DEV)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.call("glide_unet_conv3x3_wgrad_bias", d.data_ptr(), Co, a.data_ptr(), CA, b.data_ptr() if CB else None, CB, N,
              H, W, part2.data_ptr(), dw2.data_ptr(), db.data_ptr(), st)
    _lib.call("glide_unet_bias_grad", d.data_ptr(), P, Co, part2.data_ptr(), db2.data_ptr(), st)
    assert torch.equal(dw, dw2) and torch.equal(db, db2)
    x = np.concatenate([xa, xb], -1)
    ref = U.conv3x3_wgrad(dz, x)
    mag = U.conv3x3_wgrad(np.abs(dz), np.abs(x))
    got = dw.cpu().numpy().reshape(9, Co, Ci)
    assert np.all(np.abs(got - ref) <= (P + 2) * 2.0 ** -24 * mag)
