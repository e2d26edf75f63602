"""GPU parity of the ordered backward at the edges of its work items: lists of
one entry, of a batch of 64, around a segment of 128 entries and around the 16
segments that the join loads at once, with particles on both sides of the
absorption (0.3) up to which exp(-x) - 1 is summed as a series.  Reference and
bar as in the backward's other tests: the oracle's FP64 adjoint on the forward's
float32 state, |g_gpu - g_64| <= 1e-3 * (|g_64| + 1e-4 * max|g_64|).
"""
import numpy as np
import pytest

import pyoracle as O
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


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 2047, 2049])
def test_ordered_backward_edges(R, n):
    import splotch_amd as S
    print("case ordered backward edges n", n, flush=True)
    rng = np.random.default_rng(7300 + n)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    side, pal = 24, synth.default_palette()
    # footprints wider than the image: every block's list holds every particle
    view = synth.View((50.0, 50.0, -150.0), (50.0, 50.0, 50.0), (0.0, 1.0, 0.0), side, side, 3.0)
    inten = rng.lognormal(0.0, 2.5, n)
    fld = synth.Field(f32(rng.uniform(48, 52, n)), f32(rng.uniform(48, 52, n)),
                      f32(rng.uniform(48, 52, n)), f32(rng.uniform(12, 20, n)), f32(inten),
                      f32(rng.uniform(0.0, 1.0, n)))
    p, _ = O.frozen_model(fld, view, [pal], a_eq_e=False)
    fld.inten[:] = f32(inten * 0.3 / np.median(p.e0))
    p, perm = O.frozen_model(fld, view, [pal], a_eq_e=False)
    if n > 60:
        assert (p.e0 > 0.3).any() and (p.e0 < 0.3).any()
    G = rng.normal(0.0, 1.0, (side, side, 3))
    state = {"sx": p.x, "sy": p.y, "r": p.r, "e0": p.e0, "e1": p.e1, "e2": p.e2}
    gro = O.adjoint64(p, {k: v.astype(np.float64) for k, v in state.items()}, G, side, side,
                      a_eq_e=False)
    pic = torch.empty(side * side * 3, dtype=torch.float32, device="cuda")
    R.render(S.to_device(fld), S.camera_setup(view), S.params(a_eq_e=False), pic)
    out = R.backward(torch.from_numpy(f32(G).reshape(-1)).cuda(), n, screen=True)
    got = out["screen"].cpu().numpy()
    for j, k in enumerate(state):
        ref = np.zeros(n)
        ref[perm] = gro[k]
        err = np.abs(got[:, j] - ref) / (np.abs(ref) + 1e-4 * max(np.abs(ref).max(), 1e-300))
        assert err.max() <= 1e-3, (k, float(err.max()))
