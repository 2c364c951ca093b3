"""Bias and head-weight gradients: the LDS-staged kernels (16-byte aligned
tensors, channel counts that are multiples of 8) add the same values in the
same order as the per-channel kernels, which the same call reaches with a
tensor that is 2 bytes off alignment.  Equal bits, at the edges of a staged
tile (256 pixels), of a chunk (4096) and of a 64-channel group."""
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


def _bf16(n, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn(n, generator=g, device=DEV).to(torch.bfloat16).view(torch.int16)


def _off_alignment(x):
    y = torch.zeros(x.numel() + 1, dtype=torch.int16, device=DEV)
    y[1:] = x
    return y[1:]


@pytest.mark.parametrize("P", [1, 255, 256, 257, 4096, 4097, 9000])
@pytest.mark.parametrize("C", [8, 32, 64, 72, 96])
def test_bias_grad_staged_equals_per_channel(P, C):
    dz = _bf16(P * C, P + C)
    part = torch.empty(_lib.fn("glide_unet_bias_chunks")(P) * C, device=DEV)
    out = []
    for t in (dz, _off_alignment(dz)):
        db = torch.empty(C, device=DEV)
        _lib.call("glide_unet_bias_grad", t.data_ptr(), P, C, part.data_ptr(), db.data_ptr(), _st())
        out.append(db)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("P", [1, 256, 257, 4097])
@pytest.mark.parametrize("C,NO", [(8, 1), (32, 3), (64, 3), (64, 4)])
def test_head_weight_grad_staged_equals_per_entry(P, C, NO):
    x = _bf16(P * C, P)
    g = torch.Generator(device=DEV)
    g.manual_seed(C + NO)
    dout = torch.randn(P * NO, generator=g, device=DEV)
    wh = torch.randn(NO * C, generator=g, device=DEV)
    nk = NO * C + NO
    part = torch.empty(_lib.fn("glide_unet_bias_chunks")(P) * nk, device=DEV)
    out = []
    for t in (x, _off_alignment(x)):
        dx, dw = torch.empty(P * C, device=DEV), torch.empty(nk, device=DEV)
        _lib.call("glide_unet_head_bwd", dout.data_ptr(), t.data_ptr(), P, C, NO, wh.data_ptr(), dx.data_ptr(),
                  part.data_ptr(), dw.data_ptr(), _st())
        out.append((dx, dw))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
