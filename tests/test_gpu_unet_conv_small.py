"""3x3 convolutions and data gradients of batches of small or narrow images: the kernel
chosen for them against the direct one (which a bias or gradient off 16-byte alignment
takes), bit for bit, and not many times slower: tiles of 32 columns that such images leave
all but empty once took up to 25 times as long.  Both sides of the choice: whole tiles,
images of one pixel, row and column, fewer workgroups than CUs and more."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402

DEV = torch.device("cuda")


def _bits(n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(n, device=DEV, generator=g).to(torch.bfloat16).view(torch.int16)


def _time(fn):
    fn()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    for _ in range(10):
        fn()
    b.record()
    torch.cuda.synchronize()
    return a.elapsed_time(b)


@pytest.mark.parametrize("N,H,W", [(64, 1, 1), (4000, 1, 1), (4000, 2, 2), (1000, 8, 8), (500, 12, 12), (300, 500, 1),
                                   (300, 1, 500), (300, 17, 33), (40, 64, 64)])
@pytest.mark.parametrize("CA,CB,Co", [(32, 0, 32), (64, 0, 64), (96, 0, 96), (64, 64, 64), (96, 96, 96)])
def test_small_images_same_bits_as_direct(N, H, W, CA, CB, Co):
    n, Ci = N * H * W, CA + CB
    st = torch.cuda.current_stream().cuda_stream
    xa, xb, dz = _bits(n * CA, 1), (_bits(n * CB, 2) if CB else None), _bits(n * Co, 3)
    wm = torch.randn(9 * Co * Ci, device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)) * 0.05
    wb, wf = (torch.empty(wm.numel(), dtype=torch.int16, device=DEV) for _ in range(2))
    _lib.call("glide_unet_prep_weights", wm.data_ptr(), Co, Ci, wb.data_ptr(), wf.data_ptr(), st)
    bias = torch.randn(Co + 1, device=DEV)
    bias[1:] = bias[:-1].clone()
    pb = xb.data_ptr() if CB else None
    res = []
    for off in (0, 1):   # off: bias and gradients 4 bytes past 16-byte alignment
        out = torch.zeros(n * Co, dtype=torch.int16, device=DEV)
        ga, gb = torch.zeros(n * CA + off, device=DEV), torch.zeros(n * CB + off + 1, device=DEV)
        b = torch.cat([torch.zeros(off, device=DEV), bias[:Co]])[off:]
        assert (b.data_ptr() & 15) == 4 * off and (ga[off:].data_ptr() & 15) == 4 * off

        def conv():
            _lib.call("glide_unet_conv3x3", xa.data_ptr(), CA, pb, CB, N, H, W, wb.data_ptr(), Co, b.data_ptr(), 1,
                      out.data_ptr(), st)

        def dgrad():
            _lib.call("glide_unet_conv3x3_dgrad", dz.data_ptr(), Co, N, H, W, wf.data_ptr(), CA, ga[off:].data_ptr(), 0,
                      CB, gb[off:].data_ptr() if CB else None, 0, st)

        t = _time(conv), _time(dgrad)
        res.append((out.clone(), ga[off:].clone(), gb[off:off + n * CB].clone(), t))
    for k in range(3):
        assert torch.equal(res[0][k], res[1][k])
    for t, direct in zip(res[0][3], res[1][3]):
        assert t < 3.0 * direct, (t, direct)
