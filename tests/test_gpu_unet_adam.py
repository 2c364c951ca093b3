"""One optimiser step of many tensors in a launch (glide_unet_adam_items) against the
per-tensor step and weight copies: the same bits.  Tensors that end at, before and past a
block of 256 values; more tensors than one launch takes; with and without BF16 copies."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402


@pytest.mark.parametrize("wd", [0.0, 0.01])
@pytest.mark.parametrize("n_plain", [1, 31, 40])
def test_items_step_same_bits(n_plain, wd):
    gen = torch.Generator(device="cuda").manual_seed(n_plain)
    shapes = [(32, 32), (64, 32), (1, 3)]
    sizes = [9 * co * ci for co, ci in shapes] + [(1, 3, 255, 256, 257, 1000)[k % 6] for k in range(n_plain)]
    t0 = [[torch.randn(n, generator=gen, device="cuda") for _ in range(4)] for n in sizes]
    for q in t0:
        q[3].abs_()
    copies = lambda: [[torch.zeros(n, dtype=torch.int16, device="cuda") for _ in range(2)] for n in sizes[:3]]  # noqa: E731
    st = torch.cuda.current_stream().cuda_stream
    ref, ref_b = [[t.clone() for t in q] for q in t0], copies()
    for (w, g, m, v), n in zip(ref, sizes):
        _lib.call("glide_unet_adam", w.data_ptr(), g.data_ptr(), m.data_ptr(), v.data_ptr(), n, 1e-3, 0.9, 0.999, 1e-8, 3, wd, st)
    for q, (co, ci) in enumerate(shapes):
        _lib.call("glide_unet_prep_weights", ref[q][0].data_ptr(), co, ci, ref_b[q][0].data_ptr(), ref_b[q][1].data_ptr(), st)
    out, out_b = [[t.clone() for t in q] for q in t0], copies()
    items = (_lib.GlideAdamItem * len(sizes))()
    for q, n in enumerate(sizes):
        items[q] = _lib.GlideAdamItem(*(t.data_ptr() for t in out[q]), n)
        if q < 3:
            items[q].wb, items[q].wflip = (t.data_ptr() for t in out_b[q])
            items[q].cout, items[q].cin = shapes[q]
    _lib.call("glide_unet_adam_items", ctypes.byref(items), len(sizes), 1e-3, 0.9, 0.999, 1e-8, 3, wd, st)
    torch.cuda.synchronize()
    for a, b in zip(ref + ref_b, out + out_b):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
    items[0].cin = 31
    with pytest.raises(_lib.GlideError):
        _lib.call("glide_unet_adam_items", ctypes.byref(items), len(sizes), 1e-3, 0.9, 0.999, 1e-8, 3, wd, st)
