"""GPU parity of long ordered lists walked in segments.

From 160M (block, particle) entries on, an ordered pass walks its lists of
81920 entries and more in segments that start from 0 a warm-up before their
first entry; a segment whose warm-up did not reach the serial chain's state is
walked again from it.  Every footprint here covers the whole 256^2 image, so
each of its 1024 blocks has the same 160k entries, in depth order.  Bar:
bit-exact against the walk of whole lists (no producer/consumer workgroups, no
staging), with absorption that forgets a list's start within a few thousand
entries, within nearly the longest warm-up and not at all (no cut), with
absorption in one channel only, with absorption almost only where the lists are
sampled (every segment is walked again), with a list continued from an earlier
chunk, and with non-finite particles.
"""
import numpy as np
import pytest

from splotch_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N, SIDE, LEAST = 160_000, 256, 160_000_000


@pytest.fixture(scope="module")
def R():
    import splotch_amd as S
    assert torch.cuda.is_available(), "GPU test without a GPU"
    r = S.Renderer(0)
    yield r
    torch.cuda.synchronize()
    r.close()


def curtain(kind, n):
    """n particles behind each other, each wider than the image."""
    rng = np.random.default_rng(7100)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    depth = np.linspace(45.0, 55.0, n)
    inten = rng.lognormal(0.0, 0.5, n)
    if kind == "sampled":  # one batch of 64 in 2048, as the lists are sampled
        rank = np.arange(n)[::-1]  # (lists run from the far side)
        inten = np.where((rank % 2048 >= 992) & (rank % 2048 < 1056), 1.0, 1e-4)
    x, y = rng.normal(50.0, 0.3, n), rng.normal(50.0, 0.3, n)
    shuffle = rng.permutation(n)
    fld = synth.Field(f32(x[shuffle]), f32(y[shuffle]), f32(depth[shuffle]),
                      np.full(n, 90.0, np.float32), f32(inten[shuffle]),
                      f32(rng.uniform(0.0, 1.0, n)))
    if kind == "nonfinite":
        fld.inten[[5, 60_000]] = np.inf, np.nan
    return fld


@pytest.mark.parametrize("kind,brightness", [
    ("deep", 100.0), ("slow", 8.0), ("thin", 0.1), ("one_channel", 100.0), ("sampled", 100.0),
    ("chunked", 100.0), ("nonfinite", 100.0)])
def test_segments(R, kind, brightness):
    import splotch_amd as S
    x, rgb = synth.default_palette()
    if kind == "one_channel":
        rgb = np.array(rgb, np.float32)
        rgb[:, 1:] = 0.0
    R.set_palette(0, x, rgb)
    n = 250_000 if kind == "chunked" else N
    dev, cam = S.to_device(curtain(kind, n)), S.camera_setup(synth.default_view(SIDE))
    pics = []
    for whole in (True, False):
        print("case segments", kind, "whole" if whole else "cut", flush=True)
        prm = S.params(a_eq_e=False, brightness=[brightness])
        if whole:
            prm.hip_heavy = prm.hip_stage_ordered = -1
        if kind == "chunked":  # two chunks of more than LEAST entries
            prm.hip_chunk_entries = 180_000_000
        pic = torch.empty(SIDE * SIDE * 3, dtype=torch.float32, device="cuda")
        R.render(dev, cam, prm, pic)
        torch.cuda.synchronize()
        assert R.stage_times()[1]["ordered_entries"] >= LEAST * (2 if kind == "chunked" else 1)
        pics.append(pic.cpu().numpy())
    assert np.array_equal(pics[0].view(np.uint32), pics[1].view(np.uint32)), kind
