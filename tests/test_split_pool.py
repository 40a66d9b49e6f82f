"""The pool that the split order-1 decoder's graph waves put their nodes in: the count of what was asked for must
not come round (CPU, the rule itself), and parts whose nodes find no room must decode to the same field (GPU)."""
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COUNT = r"""
#include "fz_split.h"
#include <cstdio>
// Waves of 1 to 1,024 nodes take their places until three times 2^32 have been asked for; prints the nodes that
// were given room and the first place that two waves share.
int main() {
    const uint64_t cap = fz::kPoolMax;
    fz::NodeCount used = 0;
    uint64_t given = 0, end = 0, asked = 0;
    uint32_t nn = 1;
    while (asked < 3ull << 32) {
        const fz::NodeCount before = used;
        used += nn;  // what an atomic add leaves
        asked += nn;
        const uint32_t at = fz::pool_first(before, nn, cap);
        if (at != fz::kPoolNone) {
            if (at < end || at + (uint64_t)nn > cap) return printf("shared at %u\n", at), 1;
            end = at + (uint64_t)nn;
            given += nn;
        }
        nn = nn % 1024 + 1;
    }
    printf("%llu\n", (unsigned long long)given);
    return given > cap;
}
"""


def test_full_pool_stays_full(tmp_path):
    src, exe = tmp_path / "count.cpp", tmp_path / "count"
    src.write_text(COUNT)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "falcons_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    cap = 0xF0000000
    assert cap - 1024 < int(r.stdout) <= cap


@pytest.mark.gpu
@pytest.mark.parametrize("nodes", [0, 1, 5000])
def test_parts_without_room(nodes, monkeypatch, capfd):
    import falcons_amd
    from falcons_amd import synth
    from oracle_lib import Oracle
    oracle = Oracle()
    oracle.L.fo_set_simd(1)
    data = synth.power_law((61, 70, 83), -3.0, seed=5)
    stream, _ = oracle.compress(data.copy(), oracle.config(data.shape, cmpr_algo=2, eb_mode=1, abs_eb=1e-3, rel_eb=1e-3))
    want, _ = oracle.decompress(stream, data.dtype)
    ctx = falcons_amd.Context(0)
    monkeypatch.setenv("FALCONS_DECODE_STATS", "1")
    monkeypatch.setenv("FALCONS_O1_POOL_NODES", str(nodes))
    print(f"case {nodes} nodes", flush=True)
    capfd.readouterr()
    got, _, _ = ctx.decompress_ex(np.frombuffer(stream, dtype=np.uint8), data.dtype)
    err = capfd.readouterr().err
    ctx.close()
    assert np.array_equal(got.reshape(-1).view(np.uint8), want.reshape(-1).view(np.uint8))
    m = re.search(r"walk decoded (\d+) exactly .*, (\d+) nodes of (\d+)", err)
    exact, asked, cap = (int(x) for x in m.groups())
    assert cap == nodes and asked > nodes and exact > 0, err[-2000:]
