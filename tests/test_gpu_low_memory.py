"""Frames whose staged operands do not fit the free device memory.

Staging long lists and walking them in segments are ways to be faster, so a frame
must not fail for want of their memory: with about 12 GB free, lists that need
23 GB of operands are rendered with fewer of them staged, or none, and a batch is
reserved for capture the same way.  Bar: bit-exact against the unstaged walk.
"""
import numpy as np
import pytest

from splotch_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIDE, FREE = 256, 12 << 30


@pytest.fixture
def R():
    import splotch_amd as S
    assert torch.cuda.is_available(), "GPU test without a GPU"
    r = S.Renderer(0)
    r.set_palette(0, *synth.default_palette())
    yield r
    torch.cuda.synchronize()
    r.close()


@pytest.fixture
def little_memory():
    """Holds all device memory but FREE bytes."""
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    hold = [torch.empty(free - FREE, dtype=torch.uint8, device="cuda")] if free > FREE else []
    print("free device memory: %.1f GB" % (torch.cuda.mem_get_info()[0] / 1e9), flush=True)
    yield
    hold.clear()
    torch.cuda.empty_cache()


def curtain(n):
    """n particles, each wider than the image: the same list in every block."""
    rng = np.random.default_rng(7300)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    return synth.Field(f32(rng.normal(50.0, 0.3, n)), f32(rng.normal(50.0, 0.3, n)),
                       f32(rng.uniform(45.0, 55.0, n)), np.full(n, 90.0, np.float32),
                       f32(rng.lognormal(0.0, 0.5, n)), f32(rng.uniform(0.0, 1.0, n)))


@pytest.mark.parametrize("additive", [True, False])
def test_staging_without_room(R, little_memory, additive):
    import splotch_amd as S
    n = 23_000 if additive else 10_000  # x 1296 blocks: 23 GB of operands each
    dev, cam = S.to_device(curtain(n)), S.camera_setup(synth.default_view(SIDE))
    pic = torch.empty(SIDE * SIDE * 3, dtype=torch.float32, device="cuda")
    off = S.params(a_eq_e=additive, hip_stage=-1, hip_stage_ordered=-1)
    given = S.params(a_eq_e=additive, hip_stage=4096, hip_stage_ordered=4096)
    print("case unstaged, additive", additive, flush=True)
    R.render(dev, cam, off, pic)
    torch.cuda.synchronize()
    want = pic.cpu().numpy()
    for prm in (given, S.params(a_eq_e=additive)):
        print("case staged for want of room, additive", additive, flush=True)
        pic.fill_(7.0)
        R.render(dev, cam, prm, pic)
        torch.cuda.synchronize()
        assert np.array_equal(pic.cpu().numpy().view(np.uint32), want.view(np.uint32))
    print("case reserved, additive", additive, flush=True)
    R.capture_reserve([(dev, cam, given, pic)], 1.25)
    torch.cuda.synchronize()
    assert np.array_equal(pic.cpu().numpy().view(np.uint32), want.view(np.uint32))
