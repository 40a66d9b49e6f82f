"""The order-1 tANS decoder that takes a chain from its first symbol (one workgroup a chain), against the
oracle bit for bit: chain lengths around a round of its log and its group of steps, escapes in the table
entries and on the rare path, and entries that stand for several steps (few bits a symbol)."""
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


CASES = [
    ("escapes-inline", lambda: synth.power_law((48, 50, 51), -3.0, seed=1), 1, 1e-4),
    ("escapes-rare-path", lambda: synth.power_law((64, 65, 66), -3.0, seed=2), 1, 2e-3),
    ("no-escapes", lambda: synth.power_law((301, 307), -3.0, seed=3), 1, 1e-2),
    ("front-f64", lambda: synth.front((64, 65, 67), seed=4), 0, 1e-6),
    ("runs", lambda: synth.front((96, 97, 98), seed=5), 0, 2e-7),
    ("waves", lambda: synth.sinusoids((64, 65, 63), seed=6), 0, 1e-3),
    # n codes in four chains: one round of the log holds 1,020 states, a group 6
    *[(f"tail-{r}", (lambda r=r: synth.power_law((4 * 1020 * 21 + 4 * 6 * 3 + r,), -2.0, seed=7)), 1, 3e-4)
      for r in (0, 4, 9, 16, 23)],
    *[(f"runs-tail-{r}", (lambda r=r: synth.front((61, 64, 50 + r), seed=8)), 0, 1e-6) for r in (0, 1, 2)],
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_serial_decoder(ctx, oracle, case, monkeypatch):
    name, make, mode, eb = case
    data = make()
    oc = oracle.config(data.shape, cmpr_algo=2, eb_mode=mode, abs_eb=eb, rel_eb=eb)
    stream, _ = oracle.compress(data.copy(), oc)
    want, _ = oracle.decompress(stream, data.dtype)
    monkeypatch.setenv("FALCONS_O1_SEQUENTIAL", "1")
    print(f"case {name} {data.shape} {data.dtype}", flush=True)
    got, _, _ = ctx.decompress_ex(np.frombuffer(stream, dtype=np.uint8), data.dtype)
    assert np.array_equal(got.reshape(-1).view(np.uint8), want.reshape(-1).view(np.uint8))
