"""GPU parity of the 8x8 splat's chunk sizes: chunks of fewer than four particles
read their constants and coverage one by one, larger ones by fours, and chunks
past a short batch are masked.  Bar: bit-exact against the oracle for every
hip_ppw and hip_variant, in both modes, one and three channels per item, at list
lengths around the chunk and the batch.
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


@pytest.mark.parametrize("additive", [True, False])
@pytest.mark.parametrize("n", [1, 3, 9, 63, 66, 131, 700])
def test_chunk_sizes(R, n, additive):
    import splotch_amd as S
    rng = np.random.default_rng(40 + n)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    pos = 50.0 + rng.normal(0.0, 1.5, (n, 3))
    fld = synth.Field(f32(pos[:, 0]), f32(pos[:, 1]), f32(pos[:, 2]),
                      f32(rng.uniform(0.5, 12.0, n)), f32(rng.lognormal(1.0, 2.0, n)),
                      f32(rng.uniform(0.0, 1.0, n)))
    side = 40
    view = synth.default_view(side)
    want, _ = O.host_rendering(fld, view, [synth.default_palette()], a_eq_e=additive, stable=True)
    dev, cam = S.to_device(fld), S.camera_setup(view)
    for ppw, variant in ((1, 4), (2, 4), (4, 4), (8, 4), (0, 1), (0, 2), (0, 3), (0, 0)):
        for split in (1, 1 << 30):  # one item per channel, or one of three
            print("case chunk", n, additive, "ppw", ppw, "variant", variant, "split", split,
                  flush=True)
            pic = torch.empty(side * side * 3, dtype=torch.float32, device="cuda")
            R.render(dev, cam, S.params(a_eq_e=additive, hip_ppw=ppw, hip_variant=variant,
                                        hip_split=split, hip_stage=-1, hip_stage_ordered=-1,
                                        hip_heavy=-1), pic)
            torch.cuda.synchronize()
            assert_bitexact(pic.cpu().numpy().reshape(side, side, 3), want,
                            "n %d ppw %d variant %d split %d" % (n, ppw, variant, split))
