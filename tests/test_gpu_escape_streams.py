"""The escape side streams of the order-1 coder (classes, mantissas, raw blocks): streams against the oracle byte
for byte, with escapes around a tile of 4,096 values, few and most codes escaped, and several segments."""
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


def noisy(n, every, scale):
    """A line whose every-th value jumps: about two escaped codes for each jump."""
    x = synth.power_law((n,), -2.0, seed=11)
    x[::every] += (scale * np.sin(np.arange(len(x[::every]), dtype=np.float64) ** 2)).astype(np.float32)
    return x


CASES = [
    ("none", lambda: synth.power_law((301, 307), -3.0, seed=3), 1, 1e-2),
    ("one-tile", lambda: noisy(100003, 60, 2.0), 0, 1e-3),
    ("tiles", lambda: noisy(120011, 13, 2.0), 0, 1e-3),
    ("wide", lambda: noisy(100003, 7, 30.0), 0, 1e-3),
    ("most", lambda: np.sin(np.arange(90001, dtype=np.float64) ** 2).astype(np.float32), 0, 1e-3),
    ("most-wide", lambda: (30 * np.sin(np.arange(90001, dtype=np.float64) ** 2)).astype(np.float32), 0, 1e-3),
    ("segments", lambda: synth.power_law((260, 256, 257), -2.2, seed=5), 1, 1e-4),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_escape_streams(ctx, oracle, case):
    import falcons_amd
    name, make, mode, eb = case
    data = make()
    kw = dict(cmpr_algo=2, eb_mode=mode, abs_eb=eb, rel_eb=eb)
    c = falcons_amd.falconsConfig(*data.shape)
    for k, v in kw.items():
        setattr(c.conf, k, v)
    want, _ = oracle.compress(data.copy(), oracle.config(data.shape, **kw))
    print(f"case {name} {data.shape}", flush=True)
    got = ctx.compress_ex(data.copy(), c, simd=1)[0]
    assert bytes(got) == want
