"""GPU parity of the vectorized post-processing and normalization passes at the
sizes and alignments where their forms change: image sides around the 64 x 16
tile and the 4- and 16-byte words, misaligned byte and float images (both byte
layouts, with and without the float image); particle counts around the four per
load and the block, misaligned fields, types past ptypes, vector colours.
Bar: bit-exact against the oracle (logged values one ulp, as log10 is pinned).
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


def at_offset(a, off):
    """A device tensor with a's values, `off` elements into its allocation."""
    t = torch.from_numpy(np.ascontiguousarray(a))
    d = torch.zeros(t.numel() + off, dtype=t.dtype, device="cuda")[off:]
    d.copy_(t)
    return d


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("xres,yres", [(1, 1), (3, 5), (64, 16), (65, 17), (63, 15), (80, 20),
                                       (128, 33), (52, 48), (130, 62)])
def test_post_edges(R, xres, yres, off):
    import splotch_amd as S
    rng = np.random.default_rng(xres * 100 + yres)
    pic = (-np.exp(rng.normal(-1.0, 3.0, (xres, yres, 3)))).astype(np.float32)
    pic.reshape(-1)[:: 7] = [np.nan, np.inf, -np.inf, 3e8, -0.0, 1e-3, -21.0][xres % 7]
    for a_eq_e in (True, False):
        q = S.post(a_eq_e=a_eq_e)
        want, tga = O.postprocess(pic.copy(), a_eq_e=a_eq_e)
        body = np.frombuffer(bytes(tga), np.uint8)[18:]
        for layout in (0, 1):
            for floats in (True, False):
                print("case post", xres, yres, "off", off, a_eq_e, layout, floats, flush=True)
                d = at_offset(pic.reshape(-1), off)
                out = at_offset(np.zeros(pic.size, np.float32), off) if floats else None
                rgb8 = at_offset(np.full(pic.size, 77, np.uint8), off)
                R.postprocess(d, xres, yres, q, out, rgb8, layout)
                torch.cuda.synchronize()
                got = rgb8.cpu().numpy()
                if layout == 0:  # x-major RGB -> rows of iy, B G R
                    got = got.reshape(xres, yres, 3)[:, :, ::-1].transpose(1, 0, 2).reshape(-1)
                assert np.array_equal(got, body), (layout, floats, a_eq_e)
                if floats:
                    g = out.cpu().numpy().reshape(pic.shape)
                    nan = np.isnan(want)
                    assert np.array_equal(np.isnan(g), nan)
                    assert_bitexact(np.where(nan, 0, g), np.where(nan, 0, want).astype(np.float32))


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 2047, 2048, 2051, 8193, (1 << 19) + 5])
def test_normalize_edges(R, n, off):
    import splotch_amd as S
    rng = np.random.default_rng(n)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    typ = rng.integers(0, 3, n).astype(np.uint8)  # type 2 lies past ptypes
    src = dict(inten=f32(rng.lognormal(0, 1, n)), col=f32(rng.normal(0, 2, n)),
               c1=f32(rng.uniform(0, 3, n)), c2=f32(rng.uniform(1, 2, n)),
               hsml=f32(rng.uniform(.1, 1, n)))
    for vec in (False, True):
        print("case normalize", n, "off", off, "vector", vec, flush=True)
        q = S.norm_from_par("ptypes=2\n" + ("color_is_vector1=T\n" if vec else ""))
        d = {k: at_offset(v, off) for k, v in src.items()}
        d["type"] = at_offset(typ, off)
        R.normalize(d, q, ranges=False)
        torch.cuda.synchronize()
        want = {k: src[k].copy() for k in ("inten", "col", "c1", "c2")}
        for t in range(2):
            sel = typ == t
            if not sel.any():
                continue
            for keys in (("inten",), ("col", "c1", "c2") if vec and t == 1 else ("col",)):
                lo = min(src[k][sel].min() for k in keys)
                hi = max(src[k][sel].max() for k in keys)
                for k in keys:
                    v = src[k][sel]
                    want[k][sel] = (v - lo) / (hi - lo) if hi != lo else np.float32(1)
        for k, w in want.items():
            assert_bitexact(d[k].cpu().numpy(), w, "%s n %d vec %s" % (k, n, vec))
