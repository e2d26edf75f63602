"""GPU parity of particle_normalize's logged and vector-coloured forms at their
tails: 16-byte vectors whose four particles mix types with logs, types without
and types past ptypes are written back whole, and the workgroup's size changes
at 2^20 (logs) and 2^21 particles (vector colours).  Aligned and misaligned
fields.  Bar: fields without logs and the particles of types past ptypes bit for
bit; a logged value and its type's extremes are each pinned to one ulp, so (v -
lo) / (hi - lo) to 4 ulp of the extremes over their distance, and its own rounding.
"""
import numpy as np
import pytest

import pyoracle as O
from helpers import assert_bitexact

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

FIELDS = (("I", "inten"), ("er", "col"), ("eg", "c1"), ("eb", "c2"), ("r", "hsml"))


@pytest.fixture(scope="module")
def R():
    import splotch_amd as S
    assert torch.cuda.is_available(), "GPU test without a GPU"
    r = S.Renderer(0)
    yield r
    torch.cuda.synchronize()
    r.close()


def at_offset(a, off):
    """A device tensor with a's values, `off` elements into its allocation."""
    t = torch.from_numpy(np.ascontiguousarray(a))
    d = torch.zeros(t.numel() + off, dtype=t.dtype, device="cuda")[off:]
    d.copy_(t)
    return d


LOGS = dict(intensity_log0="true", color_log0="true", color_asinh1="true")


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 5, 2049, (1 << 19) + 5, (1 << 20) - 1, (1 << 20) + 3,
                               (1 << 21) + 2])
def test_normalize_logs(R, n, off):
    import splotch_amd as S
    rng = np.random.default_rng(n)
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    src = dict(I=f32(rng.lognormal(0, 2, n)), er=f32(rng.lognormal(0, 1.5, n)),
               eg=f32(rng.lognormal(0, 1, n)), eb=f32(rng.lognormal(0, 1, n)),
               r=f32(rng.uniform(.1, 1, n)),
               type=rng.integers(0, 4, n).astype(np.uint8))  # type 3 lies past ptypes
    src["I"][::97] = -1.0
    src["er"][::89] = 0.0
    for vec in (False, True):
        kv = dict(LOGS, color_is_vector1="true") if vec else LOGS
        print("case normalize logs", n, "off", off, "vector", vec, flush=True)
        d = {dk: at_offset(src[fk], off) for fk, dk in FIELDS}
        d["type"] = at_offset(src["type"], off)
        R.normalize(d, S.norm_from_par(O.kv_text(dict(kv, ptypes=3))), ranges=False)
        torch.cuda.synchronize()
        known = src["type"] < 3
        part = {k: v[known] for k, v in src.items()}
        want, out, _ = O.normalize(part, kv, 3)
        t = part["type"]
        for fk, dk in FIELDS:
            got = d[dk].cpu().numpy()
            assert_bitexact(got[~known], src[fk][~known], "%s of a type past ptypes" % fk)
            g, w = got[known], want[fk]
            for k in range(3):
                logged = fk == "I" and k == 0 or fk == "er" and k < 2 or (
                    fk in ("eg", "eb") and vec and k == 1)
                a, b = g[t == k], w[t == k]
                if not logged or not a.size:
                    assert_bitexact(a, b, "%s of type %d, n %d" % (fk, k, n))
                    continue
                lo, hi = out[k, 4:6] if fk == "I" else out[k, 0:2]
                tol = 2.0 ** -23
                if hi > lo:
                    tol += 4.0 * np.spacing(max(abs(lo), abs(hi))) / (float(hi) - float(lo))
                assert np.abs(a.astype(np.float64) - b).max() <= tol, (fk, k, n, vec)
