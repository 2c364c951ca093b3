"""The convolution and its data gradient against the float64 oracle where the
tiling can go wrong: images smaller than a tile (2 to 8 rows x 32 columns) or
just past its edge, several images, one and several 32-channel chunks of two
inputs, the most channels that are staged in LDS (192) and counts that are
not (160, 224).

Tolerance per entry: an FP32 sum of n products in any order is off by at most
(n + 2) 2^-24 times the sum of the products' magnitudes; a BF16 output may
also round the other way, by one BF16 unit."""
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


def _f32(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(DEV)


@pytest.mark.parametrize("N,H,W", [(1, 1, 1), (2, 3, 31), (1, 8, 32), (1, 9, 33), (3, 17, 70), (1, 64, 64)])
@pytest.mark.parametrize("CA,CB,Co", [(32, 0, 32), (64, 32, 64), (96, 96, 32), (96, 64, 32), (224, 0, 32)])
def test_conv_and_data_gradient_match_oracle(N, H, W, CA, CB, Co):
    rng = np.random.default_rng(H + W + CA)
    Ci = CA + CB
    x = U.bf16(rng.standard_normal((N, H, W, Ci)).astype(np.float32))
    dz = U.bf16(rng.standard_normal((N, H, W, Co)).astype(np.float32))
    w = U.bf16((rng.standard_normal((9, Co, Ci)) * 0.1).astype(np.float32))
    b = (rng.standard_normal(Co) * 0.1).astype(np.float32)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    wb, wf = (torch.empty(w.size, dtype=torch.int16, device=DEV) for _ in range(2))
    wm, bd = _f32(w), _f32(b)
    _lib.call("glide_unet_prep_weights", wm.data_ptr(), Co, Ci, wb.data_ptr(), wf.data_ptr(), st)
    xa, xb, d = _dev(x[..., :CA]), (_dev(x[..., CA:]) if CB else None), _dev(dz)
    out = torch.empty(N * H * W * Co, dtype=torch.int16, device=DEV)
    pb = xb.data_ptr() if CB else None
    _lib.call("glide_unet_conv3x3", xa.data_ptr(), CA, pb, CB, N, H, W, wb.data_ptr(), Co, bd.data_ptr(), 0,
              out.data_ptr(), st)
    got = U.from_bits(out.cpu().numpy().view(np.uint16)).reshape(N, H, W, Co)
    ref = U.conv3x3(x, w, b, relu=False, rounding=False)
    mag = U.conv3x3(np.abs(x), np.abs(w), np.abs(b), relu=False, rounding=False)
    tol = (9 * Ci + 3) * 2.0 ** -24 * mag
    assert np.all(np.abs(got - ref) <= tol + (np.abs(ref) + tol) * 2.0 ** -8)
    ga = torch.empty(N * H * W * CA, device=DEV)
    gb = torch.full((N * H * W * max(CB, 1),), 2.0, device=DEV)
    _lib.call("glide_unet_conv3x3_dgrad", d.data_ptr(), Co, N, H, W, wf.data_ptr(), CA, ga.data_ptr(), 0, CB,
              gb.data_ptr() if CB else None, 1, st)
    ref = U.conv3x3_dgrad(dz, w)
    mag = U.conv3x3_dgrad(np.abs(dz), np.abs(w))
    got = ga.cpu().numpy().reshape(N, H, W, CA)
    if CB:
        got = np.concatenate([got, gb.cpu().numpy().reshape(N, H, W, CB)], -1)
        ref[..., CA:] += 2.0
        mag[..., CA:] += 2.0
    assert np.all(np.abs(got - ref) <= (9 * Co + 3) * 2.0 ** -24 * mag)
