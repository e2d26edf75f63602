"""GPU parity of binning and depth sort around the sizes where the scans and
radix sorts change form: one workgroup up to 4096 pairs / 16384 elements, tiles of
1024 pairs up to 131072, the
tiles' histograms summed by the scatter up to 128 tiles (524288 pairs), then
scanned; the pass sizes read late or early.  Bar: the reference-tile lists and
the render order equal the oracle's, and an ordered image (for the sizes it is
quick for) is bit-exact against the oracle.
"""
import numpy as np
import pytest

import pyoracle as O
from helpers import assert_bitexact
from splotch_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def R():
    import splotch_amd as S
    assert torch.cuda.is_available(), "GPU test without a GPU"
    r = S.Renderer(0)
    r.set_palette(0, *synth.default_palette())
    yield r
    torch.cuda.synchronize()
    r.close()


@pytest.mark.parametrize("n", [1, 2, 63, 4095, 4096, 4097, 16384, 16385, 70001, 131072,
                               131073, 140000, 524288, 540000])
def test_sort_sizes(R, n):
    import splotch_amd as S
    print("case sort sizes n", n, flush=True)
    fld = synth.plummer_field(n, 700 + n, hsml_fixed=0.02)
    view = synth.default_view(400, 300)
    pal = synth.default_palette()
    prm = S.params(a_eq_e=False)
    cam = S.camera_setup(view)
    dev = S.to_device(fld)
    off, idx, order = R.bins(dev, cam, prm, True)
    p = O.project_colorize(fld, view, [pal])
    perm = O.sort_perm(p, 1, True)
    live = perm[p.active[perm] != 0]
    assert np.array_equal(order, live.astype(np.uint32))
    q = p.take(perm)
    want_off, want_idx = O.bins(q, view.xres, view.yres, 50)
    assert np.array_equal(off, want_off)
    assert np.array_equal(idx, np.asarray(perm)[want_idx].astype(np.uint32))
    pic = torch.empty(view.xres * view.yres * 3, dtype=torch.float32, device="cuda")
    R.render(dev, cam, prm, pic)
    torch.cuda.synchronize()
    want, _ = O.host_rendering(fld, view, [pal], a_eq_e=False, stable=True)
    assert_bitexact(pic.cpu().numpy().reshape(view.xres, view.yres, 3), want, "n %d" % n)
