"""GPU parity of the staged lists' rows: a pixel's chain holds only the entries
whose footprint covers it, in batches of 64 entries, groups of 4 rows, loads of
32 rows and a ring of such loads.  Bar: bit-exact against the oracle, with every
list staged, at list lengths around each of those sizes (full coverage: as many
rows as entries), and with footprints of about a pixel (most pixels of a block
have few rows or none, columns of a block differ).
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


def cluster(n, hsml, spread, seed):
    """n particles around the box centre: `spread` box units wide."""
    rng = np.random.default_rng(seed)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    pos = 50.0 + rng.normal(0.0, spread, (n, 3))
    return synth.Field(f32(pos[:, 0]), f32(pos[:, 1]), f32(pos[:, 2]), np.full(n, hsml, np.float32),
                       f32(rng.lognormal(0.0, 1.0, n)), f32(rng.uniform(0.0, 1.0, n)))


@pytest.mark.parametrize("additive", [True, False])
@pytest.mark.parametrize("n", [1, 4, 5, 63, 64, 65, 319, 321, 1023, 1024, 1025, 1088, 2100])
def test_staged_rows(R, n, additive):
    import splotch_amd as S
    for hsml, spread, side in ((12.0, 0.5, 48), (0.05, 1.0, 64)):
        fld, view = cluster(n, hsml, spread, 900 + n), synth.default_view(side)
        print("case staged rows n", n, "additive", additive, "hsml", hsml, flush=True)
        want, _ = O.host_rendering(fld, view, [synth.default_palette()], a_eq_e=additive,
                                   stable=True)
        pic = torch.empty(side * side * 3, dtype=torch.float32, device="cuda")
        R.render(S.to_device(fld), S.camera_setup(view),
                 S.params(a_eq_e=additive, hip_stage=1, hip_stage_ordered=1), pic)
        torch.cuda.synchronize()
        assert_bitexact(pic.cpu().numpy().reshape(side, side, 3), want,
                        "n %d additive %s hsml %g" % (n, additive, hsml))
