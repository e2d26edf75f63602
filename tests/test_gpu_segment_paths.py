"""GPU test of where ordered lists are walked in segments, and beside what.

The work-item trace has a record per such list (channel code 4, 5 where some of its
segments are walked by channel), which shows that a frame took the path it is meant
to test: lists cut or not by their absorption, walks by channel, two chunks of which
the second continues cut lists from the image, lists whose samples do not represent them (walked
again by channel), cut lists beside producer/consumer
workgroups, beside staged lists, and beside an additive pass.  Bar: bit-exact against
the walk of whole lists (no producer/consumer workgroups, no staging).

At 256^2 there are 1296 8x8 blocks (of 50 px tiles); "curtain" particles cover all.
"""
import numpy as np
import pytest

from splotch_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIDE, BLOCKS, LEAST = 256, 1296, 160_000_000


@pytest.fixture(scope="module")
def R():
    import splotch_amd as S
    assert torch.cuda.is_available(), "GPU test without a GPU"
    r = S.Renderer(0)
    for t in range(2):
        r.set_palette(t, *synth.default_palette())
    yield r
    torch.cuda.synchronize()
    r.close()


def f32(a):
    return np.ascontiguousarray(a, np.float32)


def cluster(n, x, hsml, inten, spread=0.3):
    """n particles behind each other around (x, 50), in shuffled order; inten: per
    particle in list order (lists run from the far side)."""
    rng = np.random.default_rng(7200)
    fld = [rng.normal(x, spread, n), rng.normal(50.0, spread, n), np.linspace(55.0, 45.0, n),
           np.full(n, hsml), np.broadcast_to(inten, n), rng.uniform(0.0, 1.0, n)]
    k = rng.permutation(n)
    return synth.Field(*(f32(a[k]) for a in fld))


def late(n):
    """Absorption in the 34th to 40th of the samples (2048 entries) only."""
    s = np.arange(n) // 2048
    return np.where((s >= 33) & (s < 40), 1.0, 1e-4)


def sampled(n):
    """Absorption almost only where the lists are sampled."""
    s = np.arange(n) % 2048
    return np.where((s >= 992) & (s < 1056), 1.0, 1e-4)


# kind: (field, render keys, check of the ordered trace's lengths and channel codes)
def frame(kind):
    if kind == "deep":
        return cluster(160_000, 50.0, 90.0, 1.0), {}, lambda ln, ch: (ch == 4).all()
    if kind == "thin":
        return cluster(160_000, 50.0, 90.0, 1e-5), {}, lambda ln, ch: (ch <= 3).all()
    if kind == "by_channel":  # the last walk has 39 samples, one wave at most 37
        return cluster(160_000, 50.0, 90.0, late(160_000)), {}, lambda ln, ch: (ch == 5).any()
    if kind == "chunked":  # two chunks of 168.7M and 174.7M entries; the trace is the second's
        return (cluster(265_000, 50.0, 90.0, 1.0), dict(hip_chunk_entries=180_000_000),
                lambda ln, ch: (ch == 4).all() and (ln > 130_000).all() and (ln < 136_000).all())
    if kind == "sampled":  # a few long lists
        a, b = cluster(240_000, 30.0, 35.0, 1.0), cluster(500_000, 92.0, 4.0, sampled(500_000), 0.02)
        return (synth.concat(a, b), {},
                lambda ln, ch: ((ch >= 4) & (ln == 500_000)).sum() > 2 and (ch >= 4).sum() > 50)
    if kind == "sampled_chunked":  # in both chunks, the second from the image
        inten = np.concatenate([sampled(130_207), sampled(134_793)])  # the chunks' particles
        return (cluster(265_000, 50.0, 90.0, inten), dict(hip_chunk_entries=180_000_000),
                lambda ln, ch: (ln == 134_793).all() and (ch >= 4).all())
    if kind == "beside_workgroups":  # a disc of cut lists, and one of lists that cannot be
        a, b = cluster(230_000, 80.0, 20.0, 1.0), cluster(230_000, 20.0, 20.0, 1e-5)
        return (synth.concat(a, b), {},
                lambda ln, ch: (ch == 4).sum() > 50 and ((ch == 3) & (ln >= 81920)).sum() > 50)
    if kind == "beside_staged":  # a few longer lists of small particles, staged
        a = cluster(240_000, 30.0, 35.0, 1.0)
        b = cluster(700_000, 92.0, 1.2, 1e-5, 0.02)
        return (synth.concat(a, b), {},
                lambda ln, ch: (ch == 4).sum() > 50 and ((ch == 3) & (ln >= 600_000)).sum() > 1)
    assert kind == "beside_additive"
    a, b = cluster(130_000, 50.0, 90.0, 1.0), cluster(20_000, 45.0, 60.0, 1.0)
    b.type = np.ones(b.n, np.uint8)
    return (synth.concat(a, b), dict(ptypes=2, a_eq_e=[0, 1], brightness=[100.0, 1.0]),
            lambda ln, ch: (ch == 4).all())


@pytest.mark.parametrize("kind", ["deep", "thin", "by_channel", "chunked", "sampled",
                                  "sampled_chunked", "beside_workgroups", "beside_staged",
                                  "beside_additive"])
def test_segment_paths(R, kind):
    import splotch_amd as S
    fld, keys, check = frame(kind)
    if keys.get("ptypes", 1) == 1:
        fld.type = None
    dev, cam = S.to_device(fld), S.camera_setup(synth.default_view(SIDE))
    pics = []
    for whole in (True, False):
        print("case segments", kind, "whole" if whole else "cut", flush=True)
        prm = S.params(**dict(dict(a_eq_e=False, brightness=[100.0]), **keys))
        if whole:
            prm.hip_heavy = prm.hip_stage_ordered = -1
        pic = torch.empty(SIDE * SIDE * 3, dtype=torch.float32, device="cuda")
        R.set_trace(not whole)
        R.set_profiling(not whole)
        try:
            R.render(dev, cam, prm, pic)
            tr = R.trace_items(True)
        finally:
            R.set_trace(False)
            R.set_profiling(False)
        torch.cuda.synchronize()
        pics.append(pic.cpu().numpy())
    stages, counts = R.stage_times()
    entries = counts["ordered_entries"]
    assert entries >= LEAST
    if kind in ("chunked", "sampled_chunked"):
        assert entries - 180_000_000 * 15 // 16 >= LEAST
    ln, ch = (tr[:, 2] & 0xffffffff).astype(np.int64), (tr[:, 2] >> 32).astype(np.int64)
    print("%s: %d entries, codes %s, longest %d" % (
        kind, entries, {int(c): int((ch == c).sum()) for c in np.unique(ch)}, ln.max()), flush=True)
    assert np.array_equal(pics[0].view(np.uint32), pics[1].view(np.uint32)), kind
    assert check(ln, ch), kind
    if kind == "beside_staged":
        assert stages["ordered_staged"] > 0.0
    if kind == "beside_workgroups":
        assert stages["ordered_k_splat_heavy"] > 0.0


def test_autotuned_frame_keeps_its_segments(R):
    """The autotuner chooses the decomposition of the other lists; tuning a frame must
    not put its long lists back into producer/consumer workgroups."""
    import splotch_amd as S
    dev = S.to_device(frame("deep")[0])
    cam = S.camera_setup(synth.default_view(SIDE))
    pics = []
    for tune in (0, 1):
        print("case segments autotuned", tune, flush=True)
        prm = S.params(a_eq_e=False, brightness=[100.0], hip_autotune=tune, hip_region=8)
        pic = torch.empty(SIDE * SIDE * 3, dtype=torch.float32, device="cuda")
        R.render(dev, cam, prm, pic)  # (tunes)
        R.set_trace(True)
        try:
            R.render(dev, cam, prm, pic)
            codes = R.trace_items(True)[:, 2] >> 32
        finally:
            R.set_trace(False)
        torch.cuda.synchronize()
        assert R.tuning()["autotuned"] == bool(tune)
        assert (codes == 4).all() and codes.size == BLOCKS
        pics.append(pic.cpu().numpy())
    assert np.array_equal(pics[0].view(np.uint32), pics[1].view(np.uint32))
