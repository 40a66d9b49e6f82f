"""The selection of escaped codes by tiles of 4,096 at lengths around one tile and around the last thread
of one, with hits everywhere, nowhere, in single codes, and at the ends: streams against the oracle byte for
byte, and decoded fields bit for bit."""
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


def field(n, kind):
    x = synth.power_law((n,), -2.0, seed=n % 97)
    if kind == "spikes":      # unpredictable values, a few codes apart
        x[::37] += np.float32(1e4)
    elif kind == "ends":
        x[0] = x[-1] = np.float32(1e4)
    elif kind == "zeros":     # the other coder: almost no value that is not zero
        x[:] = 0
        x[n // 2] = 1
    return x


@pytest.mark.parametrize("n", [2, 17, 4095, 4097, 4096 * 21 - 1, 4096 * 21 + 2, 4096 * 21 + 15, 4096 * 21 + 18])
@pytest.mark.parametrize("kind", ["plain", "spikes", "ends", "zeros"])
def test_selected_codes(ctx, oracle, n, kind):
    import falcons_amd
    data = field(n, kind)
    kw = dict(cmpr_algo=2, eb_mode=0, abs_eb=1e-4, rel_eb=1e-4)
    c = falcons_amd.falconsConfig(n)
    for k, v in kw.items():
        setattr(c.conf, k, v)
    want, _ = oracle.compress(data.copy(), oracle.config(data.shape, **kw))
    print(f"case {kind} {n}", flush=True)
    got, _ = ctx.compress_ex(data.copy(), c, simd=1)[:2]
    assert bytes(got) == want
    field_want, _ = oracle.decompress(want, data.dtype)
    dec, _, _ = ctx.decompress_ex(np.frombuffer(want, dtype=np.uint8), data.dtype)
    assert np.array_equal(dec.reshape(-1).view(np.uint8), field_want.reshape(-1).view(np.uint8))
