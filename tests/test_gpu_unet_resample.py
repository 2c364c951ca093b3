"""The convolution with upsampling and pooling around it, and its workgroups
of 1, 2 and 3 output-channel groups, against the separate kernels around the
direct convolution (which a bias off 16-byte alignment takes), bit for bit;
the network's input features against themselves at an unaligned address."""
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


def _bits(rng, *shape):
    x = U.bf16(rng.standard_normal(shape).astype(np.float32))
    return torch.from_numpy(U.to_bits(x).view(np.int16).copy()).to(DEV)


@pytest.mark.parametrize("N,H,W", [(1, 2, 2), (2, 6, 30), (1, 8, 32), (1, 10, 34), (2, 64, 96), (4, 128, 128)])
@pytest.mark.parametrize("CA,CB,Co", [(32, 0, 32), (64, 0, 64), (32, 32, 96), (96, 0, 96), (64, 64, 128), (96, 96, 64),
                                      (96, 64, 32)])
def test_resampling_conv_same_bits(N, H, W, CA, CB, Co):
    rng = np.random.default_rng(H + W + CA + Co)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    Ci = CA + CB
    half, xb, w = _bits(rng, N, H // 2, W // 2, CA), _bits(rng, N, H, W, max(CB, 1)), _bits(rng, 9, Co, Ci)
    b = torch.from_numpy(rng.standard_normal(Co + 4).astype(np.float32)).to(DEV)
    off = torch.empty(Co + 5, device=DEV)[1:]
    off.copy_(b)
    pb = xb.data_ptr() if CB else None
    up, ref, got, got2 = (torch.zeros(N * H * W * c, dtype=torch.int16, device=DEV) for c in (CA, Co, Co, Co))
    pref, pgot, pgot2 = (torch.zeros(N * (H // 2) * (W // 2) * Co, dtype=torch.int16, device=DEV) for _ in range(3))
    _lib.call("glide_unet_up2", half.data_ptr(), N, H // 2, W // 2, CA, up.data_ptr(), st)
    _lib.call("glide_unet_conv3x3", up.data_ptr(), CA, pb, CB, N, H, W, w.data_ptr(), Co, off.data_ptr(), 1, ref.data_ptr(),
              st)
    _lib.call("glide_unet_pool2", ref.data_ptr(), N, H, W, Co, pref.data_ptr(), st)
    for bias, o, p in ((b, got, pgot), (off, got2, pgot2)):
        _lib.call("glide_unet_conv3x3_up_pool", half.data_ptr(), CA, 1, pb, CB, N, H, W, w.data_ptr(), Co, bias.data_ptr(),
                  1, o.data_ptr(), p.data_ptr(), st)
        assert torch.equal(o, ref) and torch.equal(p, pref)
    got.zero_()
    _lib.call("glide_unet_conv3x3_up_pool", up.data_ptr(), CA, 0, pb, CB, N, H, W, w.data_ptr(), Co, b.data_ptr(), 1,
              got.data_ptr(), None, st)
    assert torch.equal(got, ref)


def test_odd_sizes_are_refused():
    t = torch.zeros(4096, dtype=torch.int16, device=DEV)
    b = torch.zeros(32, device=DEV)
    for up, pool in ((1, None), (0, t.data_ptr())):
        with pytest.raises(Exception):
            _lib.call("glide_unet_conv3x3_up_pool", t.data_ptr(), 32, up, None, 0, 1, 3, 2, t.data_ptr(), 32, b.data_ptr(), 0,
                      t.data_ptr(), pool, None)


@pytest.mark.parametrize("ny,nx", [(2, 2), (5, 13), (16, 64), (33, 70)])
def test_features_at_any_address(ny, nx):
    rng = np.random.default_rng(ny * nx)
    f = [torch.from_numpy(rng.uniform(1.0, 900.0, ny * nx)).to(DEV) for _ in range(4)]
    out = torch.full((ny * nx * 32 + 16,), 77, dtype=torch.int16, device=DEV)
    out2 = torch.full((ny * nx * 32 + 16,), 77, dtype=torch.int16, device=DEV)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    a = [t.data_ptr() for t in f]
    _lib.call("glide_unet_features", *a, ny, nx, 500.0, out.data_ptr(), st)
    _lib.call("glide_unet_features", *a, ny, nx, 500.0, out2.data_ptr() + 2, st)
    n = ny * nx * 32
    assert torch.equal(out[:n], out2[1:n + 1])
    assert (out[n:] == 77).all() and (out2[n + 1:] == 77).all() and out2[0] == 77
    assert (out[:n].view(-1, 32)[:, 7:] == 0).all()
