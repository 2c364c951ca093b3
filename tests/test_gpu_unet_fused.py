"""The backward passes that go through a ReLU in one kernel give the bits of
the FP32 pass followed by glide_unet_relu_bwd: the convolution's data gradient
(both the LDS-staged kernel and, at 160 channels, the direct one), the head,
pooling added to another gradient, and upsampling."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402

DEV = torch.device("cuda")


def _st():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _bf16(n, seed):
    return torch.randn(n, generator=_gen(seed), device=DEV).to(torch.bfloat16).view(torch.int16)


def _f32(n, seed):
    return torch.randn(n, generator=_gen(seed), device=DEV)


def _relu_bwd(dy, y):
    dz = torch.empty_like(y)
    _lib.call("glide_unet_relu_bwd", dy.data_ptr(), y.data_ptr(), y.numel(), dz.data_ptr(), _st())
    return dz


@pytest.mark.parametrize("N,H,W", [(1, 1, 1), (2, 9, 33), (1, 64, 64)])
@pytest.mark.parametrize("Co,Ci", [(32, 32), (96, 64), (160, 32)])
def test_conv_dgrad_relu(N, H, W, Co, Ci):
    P = N * H * W
    dz, y = _bf16(P * Co, 1), _bf16(P * Ci, 2)
    wf = _bf16(9 * Ci * Co, 3)
    ga, out = torch.empty(P * Ci, device=DEV), torch.empty(P * Ci, dtype=torch.int16, device=DEV)
    _lib.call("glide_unet_conv3x3_dgrad", dz.data_ptr(), Co, N, H, W, wf.data_ptr(), Ci, ga.data_ptr(), 0, 0, None, 0,
              _st())
    _lib.call("glide_unet_conv3x3_dgrad_relu", dz.data_ptr(), Co, N, H, W, wf.data_ptr(), Ci, y.data_ptr(),
              out.data_ptr(), _st())
    assert torch.equal(out, _relu_bwd(ga, y))


@pytest.mark.parametrize("P,C,NO", [(1, 8, 1), (300, 32, 3), (4100, 64, 4), (77, 48, 2)])
def test_head_bwd_relu(P, C, NO):
    x, dout, wh = _bf16(P * C, 4), _f32(P * NO, 5), _f32(NO * C, 6)
    nk = NO * C + NO
    part = torch.empty(_lib.fn("glide_unet_bias_chunks")(P) * nk, device=DEV)
    dx, dw, dw2 = torch.empty(P * C, device=DEV), torch.empty(nk, device=DEV), torch.empty(nk, device=DEV)
    dz = torch.empty(P * C, dtype=torch.int16, device=DEV)
    _lib.call("glide_unet_head_bwd", dout.data_ptr(), x.data_ptr(), P, C, NO, wh.data_ptr(), dx.data_ptr(),
              part.data_ptr(), dw.data_ptr(), _st())
    _lib.call("glide_unet_head_bwd_relu", dout.data_ptr(), x.data_ptr(), P, C, NO, wh.data_ptr(), dz.data_ptr(),
              part.data_ptr(), dw2.data_ptr(), _st())
    assert torch.equal(dz, _relu_bwd(dx, x)) and torch.equal(dw, dw2)


@pytest.mark.parametrize("N,H,W,C", [(1, 2, 2, 8), (2, 6, 10, 96), (1, 34, 18, 32)])
def test_pool_and_up_bwd_relu(N, H, W, C):
    n = N * H * W * C
    y, g, dy = _bf16(n, 7), _f32(n, 8), _f32(n // 4, 9)
    acc, dz = g.clone(), torch.empty(n, dtype=torch.int16, device=DEV)
    _lib.call("glide_unet_pool2_bwd", dy.data_ptr(), N, H, W, C, acc.data_ptr(), 1, _st())
    _lib.call("glide_unet_pool2_bwd_relu", dy.data_ptr(), g.data_ptr(), N, H, W, C, y.data_ptr(), dz.data_ptr(), _st())
    assert torch.equal(dz, _relu_bwd(acc, y))
    du, gu = _f32(4 * n, 10), torch.empty(n, device=DEV)
    _lib.call("glide_unet_up2_bwd", du.data_ptr(), N, H, W, C, gu.data_ptr(), _st())
    _lib.call("glide_unet_up2_bwd_relu", du.data_ptr(), N, H, W, C, y.data_ptr(), dz.data_ptr(), _st())
    assert torch.equal(dz, _relu_bwd(gu, y))
