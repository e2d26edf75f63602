"""GPU test of the long lists' rules where every particle covers every block.

Such a view has hundreds of lists as long as the longest, so that none of them
outlasts the pass and what is done for single long lists costs more than it saves:
they are not staged, and where they fill the GPU not walked by channel, while the
one long list among short ones is staged.  The stage times and the work-item trace
show the route; the images are the oracle's bit for bit.
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


def field(n, hsml, spread, seed=3):
    rng = np.random.default_rng(seed)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    pos = 50.0 + rng.normal(0.0, spread, (n, 3))
    return synth.Field(f32(pos[:, 0]), f32(pos[:, 1]), f32(pos[:, 2]), np.full(n, hsml, np.float32),
                       f32(rng.lognormal(0.0, 0.5, n)), f32(rng.uniform(0.0, 1.0, n)))


@pytest.mark.parametrize("additive", [True, False])
@pytest.mark.parametrize("kind,n,hsml,spread,side", [
    ("uniform", 2000, 90.0, 0.3, 256), ("uniform", 8000, 90.0, 0.3, 128),
    ("single", 8000, 0.3, 0.3, 256)])
def test_uniform_lists(R, kind, n, hsml, spread, side, additive):
    import splotch_amd as S
    fld, view = field(n, hsml, spread), synth.default_view(side)
    print("case lists", kind, n, "additive", additive, flush=True)
    want, _ = O.host_rendering(fld, view, [synth.default_palette()], a_eq_e=additive, stable=True)
    dev, cam = S.to_device(fld), S.camera_setup(view)
    prm = S.params(a_eq_e=additive)
    pic = torch.empty(side * side * 3, dtype=torch.float32, device="cuda")
    R.set_profiling(True)
    R.set_trace(True)
    try:
        R.render(dev, cam, prm, pic)
        tr = R.trace_items(not additive)
        stages, _ = R.stage_times()
    finally:
        R.set_profiling(False)
        R.set_trace(False)
    torch.cuda.synchronize()
    staged = stages["additive_staged" if additive else "ordered_staged"] > 0.0
    assert staged == (kind == "single")
    if kind == "uniform" and side == 256:  # (324 lists leave CUs free)
        assert (tr[:, 2] >> 32 == 3).all()
    assert_bitexact(pic.cpu().numpy().reshape(side, side, 3), want, kind)
    # the same from a reservation, whose partition is made on the device
    pic.fill_(7.0)
    R.capture_reserve([(dev, cam, prm, pic)], 1.25)
    torch.cuda.synchronize()
    assert_bitexact(pic.cpu().numpy().reshape(side, side, 3), want, kind + " reserved")


@pytest.mark.parametrize("additive", [True, False])
def test_more_than_the_workgroups_serve(R, additive):
    """1296 lists for 192 producer/consumer workgroups: the ordered ones that are
    left go by channel, the additive ones do not."""
    import splotch_amd as S
    side = 256
    fld, view = field(6000, 90.0, 0.3), synth.default_view(side)
    print("case left lists additive", additive, flush=True)
    want, _ = O.host_rendering(fld, view, [synth.default_palette()], a_eq_e=additive, stable=True)
    dev, cam = S.to_device(fld), S.camera_setup(view)
    prm = S.params(a_eq_e=additive, hip_heavy=4096)
    pic = torch.empty(side * side * 3, dtype=torch.float32, device="cuda")
    R.set_trace(True)
    try:
        R.render(dev, cam, prm, pic)
        tr = R.trace_items(not additive)
    finally:
        R.set_trace(False)
    torch.cuda.synchronize()
    assert ((tr[:, 2] >> 32) < 3).any() == (not additive)
    assert_bitexact(pic.cpu().numpy().reshape(side, side, 3), want, "left lists")
    pic.fill_(7.0)
    R.capture_reserve([(dev, cam, prm, pic)], 1.25)
    torch.cuda.synchronize()
    assert_bitexact(pic.cpu().numpy().reshape(side, side, 3), want, "left lists reserved")
