"""The split order-1 decoder where a graph is not whole: each size class of its graphs with full tables of nodes (such
parts are decoded one after another by the walk) and with all or most nodes left to the walk to read from memory,
against the oracle bit for bit. The decoder's statistics say that the class and the path were the ones meant."""
import re

import numpy as np
import pytest

from oracle_lib import Oracle
from test_gpu_split import CASES

pytestmark = pytest.mark.gpu

FIELDS = {c[0]: c[1:4] for c in CASES}
# field, size class of all its chains
CLASSES = [("few-escapes-long", 0), ("some-escapes", 1), ("spikes", 1), ("many-escapes-f64", 2), ("many-escapes", 2)]


@pytest.fixture(scope="module")
def ctx():
    import falcons_amd
    c = falcons_amd.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def streams():
    o = Oracle()
    o.L.fo_set_simd(1)
    made = {}

    def get(name):
        if name not in made:
            make, mode, eb = FIELDS[name]
            data = make()
            stream, _ = o.compress(data.copy(), o.config(data.shape, cmpr_algo=2, eb_mode=mode, abs_eb=eb, rel_eb=eb))
            made[name] = (np.frombuffer(stream, dtype=np.uint8), data.dtype, o.decompress(stream, data.dtype)[0])
        return made[name]

    return get


@pytest.mark.parametrize("switch,nodes", [(None, 0), ("FALCONS_O1_GRAPH_NODES", 0), ("FALCONS_O1_GRAPH_NODES", 20),
                                          ("FALCONS_O1_STAGE_NODES", 0), ("FALCONS_O1_STAGE_NODES", 7)])
@pytest.mark.parametrize("name,cls", CLASSES, ids=[c[0] for c in CLASSES])
def test_split_paths(ctx, streams, monkeypatch, capfd, name, cls, switch, nodes):
    stream, dtype, want = streams(name)
    monkeypatch.setenv("FALCONS_O1_PARALLEL_SHORT", "1")
    monkeypatch.setenv("FALCONS_DECODE_STATS", "1")
    if switch:
        monkeypatch.setenv(switch, str(nodes))
    capfd.readouterr()
    print(f"case {name} {switch} {nodes}", flush=True)
    got, _, _ = ctx.decompress_ex(stream, dtype)
    err = capfd.readouterr().err
    assert np.array_equal(got.reshape(-1).view(np.uint8), want.reshape(-1).view(np.uint8))
    chains = [int(c) for c in re.findall(r" \d+:\d+/\d+/esc\d+/b[\d.]+/s\d+/h\d+/c(\d+)", err)]
    assert chains == [cls] * 4, err[-2000:]
    parts, exact, lost, used = (int(x) for x in re.search(
        r"split chains, (\d+) parts, walk decoded (\d+) exactly \((\d+) without a whole path, .*, (\d+) nodes of \d+",
        err).groups())
    if switch == "FALCONS_O1_GRAPH_NODES":
        waves = parts * 3  # at most: a part a wave, three rounds
        assert used <= nodes * waves and lost > 0
        assert exact > (parts // 2 if nodes == 0 else 20)
    else:
        assert used > 1000 and exact < parts // 20  # the escapes' edges are in the graphs
