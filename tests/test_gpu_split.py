"""The split order-1 tANS decoder (warm-up, graphs, walk, output) at the sizes where it can go wrong,
against the oracle bit for bit: chains just above and below its shortest, parts that end with the
chain, each size class of its graphs, and chains whose sets or graphs lack the true path."""
import re

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


def counts(shape, seed, scale):
    return (4000 + scale * synth.power_law(shape, -3.0, seed=seed)).round().astype(np.int32)


# name, field, mode, bound, whether its chains are split; a chain holds a quarter of the field's codes
# (fields of much fewer than 85,000 codes take the other coder)
CASES = [
    ("shortest", lambda: synth.power_law((33, 40, 65), -3.0, seed=1), 1, 1e-3, True),
    ("line", lambda: synth.power_law((150001,), -2.0, seed=2), 1, 1e-3, True),
    ("few-escapes", lambda: synth.power_law((64, 65, 67), -3.0, seed=3), 1, 1e-2, True),
    ("few-escapes-long", lambda: synth.power_law((1025, 1031), -3.0, seed=4), 1, 1e-3, True),
    ("some-escapes", lambda: synth.power_law((61, 70, 83), -3.0, seed=5), 1, 1e-3, True),
    ("many-escapes-f64", lambda: synth.power_law((90, 67, 71), -3.0, seed=6, dtype=np.float64), 1, 7e-4, True),
    ("many-escapes", lambda: counts((61, 64, 75), 7, 600), 0, 4.0, True),
    ("most-escapes", lambda: counts((61, 64, 75), 8, 1400), 0, 4.0, False),
    ("spikes", lambda: np.where(np.arange(64 * 65 * 66).reshape(64, 65, 66) % 389 == 0, np.float32(3),
                                synth.power_law((64, 65, 66), -3.0, seed=9)), 1, 1e-3, True),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_split_decoder(ctx, oracle, case, monkeypatch, capfd):
    import falcons_amd
    name, make, mode, eb, split = case
    data = make()
    oc = oracle.config(data.shape, cmpr_algo=2, eb_mode=mode, abs_eb=eb, rel_eb=eb)
    stream, _ = oracle.compress(data.copy(), oc)
    want, _ = oracle.decompress(stream, data.dtype)
    monkeypatch.setenv("FALCONS_O1_PARALLEL_SHORT", "1")
    monkeypatch.setenv("FALCONS_DECODE_STATS", "1")
    capfd.readouterr()
    print(f"case {name} {data.shape} {data.dtype}", flush=True)
    got, _, _ = ctx.decompress_ex(np.frombuffer(stream, dtype=np.uint8), data.dtype)
    err = capfd.readouterr().err
    assert np.array_equal(got.reshape(-1).view(np.uint8), want.reshape(-1).view(np.uint8))
    assert bool(re.search(r"\[o1 decode\] \d+ split chains", err)) == split, err[-2000:]
