"""The order-1 encoder's pieces for short arrays (sets of states and a walk) against the oracle byte for byte:
last pieces of one step and of a whole piece, chains around the longest it takes, few and many bits a
symbol, and codes whose symbols are all too frequent for sets, which the other pieces then code."""
import numpy as np
import pytest

from falcons_amd import synth
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import falcons_amd
    c = falcons_amd.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def oracle():
    o = Oracle()
    o.L.fo_set_simd(1)
    return o


def binary(n):
    return np.random.default_rng(3).integers(0, 2, n).astype(np.float32)


# name, field, mode, bound, whether the other pieces code it (None: not said)
CASES = [
    # a chain holds a quarter of the codes, a piece 256 steps
    *[(f"line-{r}", (lambda r=r: synth.power_law((4 * 256 * 90 + r,), -2.0, seed=2)), 1, 1e-5, False)
      for r in (0, 24, 28, 32, 36, 1020, 1052)],
    ("few-bits", lambda: synth.power_law((64, 65, 67), -3.0, seed=3), 1, 1e-2, False),
    ("many-bits", lambda: synth.power_law((61, 70, 83), -3.0, seed=5), 1, 1e-3, False),
    ("escapes", lambda: synth.power_law((61, 70, 83), -3.0, seed=5), 1, 1e-4, False),
    ("two-values", lambda: binary(100003), 0, 1 / 32, None),
    ("frequent", lambda: synth.power_law((92160,), -2.0, seed=2), 1, 1e-3, True),
    ("longest", lambda: synth.power_law((7 << 19,), -2.0, seed=4), 1, 1e-5, False),
    ("too-long", lambda: synth.power_law(((7 << 19) + 40000,), -2.0, seed=4), 1, 1e-5, True),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_encoder_sets(ctx, oracle, case):
    import falcons_amd
    name, make, mode, eb, other = case
    data = make()
    kw = dict(cmpr_algo=2, eb_mode=mode, abs_eb=eb, rel_eb=eb)
    c = falcons_amd.falconsConfig(*data.shape)
    for k, v in kw.items():
        setattr(c.conf, k, v)
    want, _ = oracle.compress(data.copy(), oracle.config(data.shape, **kw))
    print(f"case {name} {data.shape}", flush=True)
    ctx.profile(True)
    ctx.profile_reset()
    got = ctx.compress_ex(data.copy(), c, simd=1)[0]
    k = ctx.kernel_times()
    ctx.profile(False)
    assert bytes(got) == want
    assert other is None or ("o1_encode_fix" in k) == other, sorted(k)
