"""The FSE coder of class bytes (tables, sets of states, walk, bits) against the oracle byte for byte: streams of one
symbol more and less than a load, a noted state, a piece and a block, with rare, common and equally frequent
symbols (no two of their states ever meet: the walk runs those pieces itself)."""
import numpy as np
import pytest

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


SYMBOLS = {
    "two": ([3, 12], [0.5, 0.5]),
    "rare": ([3, 12, 50], [0.985, 0.01, 0.005]),
    "falling": ([1, 3, 6, 12, 25, 50, 100, 200, 400], [0.5, 0.25, 0.12, 0.06, 0.03, 0.02, 0.01, 0.007, 0.003]),
}


def spikes(nv, kind):
    """A line of zeros with nv values at odd places: the finest level codes them as they are, in their order."""
    rng = np.random.default_rng(nv)
    val, p = SYMBOLS[kind]
    x = np.zeros(12 * nv + 30, np.float32)
    x[1:12 * nv:12] = rng.choice(np.array(val, np.float32), nv, p=p) * rng.choice(np.array([-2, 2], np.float32), nv)
    return x


@pytest.mark.parametrize("nv", [1, 2, 3, 4, 17, 255, 258, 259, 1025, 1026, 1027, 5122, 65535, 65536, 65537, 131075])
@pytest.mark.parametrize("kind", list(SYMBOLS))
def test_fse_blocks(ctx, oracle, nv, kind):
    import falcons_amd
    data = spikes(nv, kind)
    kw = dict(cmpr_algo=2, eb_mode=0, abs_eb=1.0, rel_eb=1.0)
    c = falcons_amd.falconsConfig(*data.shape)
    for k, v in kw.items():
        setattr(c.conf, k, v)
    want, _ = oracle.compress(data.copy(), oracle.config(data.shape, **kw))
    print(f"case {kind} {nv}", flush=True)
    got = ctx.compress_ex(data.copy(), c, simd=1)[0]
    assert bytes(got) == want
