"""GPU test of hip_split: lists from that length on which are neither staged nor a
producer/consumer workgroup's are walked as three one-channel items, also where
the staging rule stages longer lists only.  The work-item trace shows them; the
image is the default's bit for bit, plain and replayed from a captured
device-count render.
"""
import math

import numpy as np
import pytest

from splotch_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIDE = 512


@pytest.fixture(scope="module")
def R():
    import splotch_amd as S
    assert torch.cuda.is_available(), "GPU test without a GPU"
    r = S.Renderer(0)
    r.set_palette(0, *synth.default_palette())
    yield r
    torch.cuda.synchronize()
    r.close()


@pytest.mark.parametrize("additive,split", [(False, 512), (False, 300), (False, 100), (True, 256)])
def test_split_of_unstaged_lists(R, additive, split):
    """1M particles, 3.9M entries: lists are staged from about 2900 (additive) and
    5500 entries on, and by default walked by channel from 1448 on."""
    import splotch_amd as S
    fld = synth.plummer_field(1_000_000, 1100, hsml_mu=math.log(0.5), ptype=0)
    dev, cam = S.to_device(fld), S.camera_setup(synth.default_view(SIDE))
    pic = torch.empty(SIDE * SIDE * 3, dtype=torch.float32, device="cuda")
    print("case split", split, "additive", additive, flush=True)
    R.render(dev, cam, S.params(a_eq_e=additive, brightness=[0.5]), pic)
    torch.cuda.synchronize()
    want = pic.cpu().numpy()
    prm = S.params(a_eq_e=additive, brightness=[0.5], hip_split=split)
    R.set_trace(True)
    try:
        R.render(dev, cam, prm, pic)
        tr = R.trace_items(not additive)
    finally:
        R.set_trace(False)
    torch.cuda.synchronize()
    assert np.array_equal(pic.cpu().numpy().view(np.uint32), want.view(np.uint32))
    ln, ch = (tr[:, 2] & 0xffffffff).astype(np.int64), tr[:, 2] >> 32
    least = split * 2 if additive else split  # 256 x 2^(j/2) above 256: 512, 300 -> 256, 512
    least = 256 if least == 300 else least
    sel = (ln >= least * 1.2) & (ln < 1448)  # (the levels' order is by quarter octaves)
    for c in range(3):
        assert (ch[sel] == c).sum() * 3 == sel.sum() > 0, "lists %d to 1448 by channel" % least
    assert (ch[(ln > 0) & (ln < least * 0.8)] == 3).all()
    R.capture_reserve([(dev, cam, prm, pic)], 1.25)
    torch.cuda.synchronize()
    assert np.array_equal(pic.cpu().numpy().view(np.uint32), want.view(np.uint32))
