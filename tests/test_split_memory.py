"""Device memory of the split order-1 decoder: the plans' bytes and the choice of chains (CPU, the rules themselves),
and on the GPU the workspace that a call holds, calls with less memory than they ask for, and requests whose
budget leaves the split decoder little or nothing."""
import os
import re
import subprocess

import numpy as np
import pytest

from falcons_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PLANS = r"""
#include "fz_split.h"
#include <cstdio>
#include <cstdlib>
using namespace fz;
#define CHECK(c, ...) if (!(c)) { printf(#c ": " __VA_ARGS__); printf("\n"); exit(1); }
static double pi[kO1Ctx];
static int16_t norm[kO1Ctx * kO1Sym];
static SplitPlan plan(uint64_t m, double bits, int escape, uint64_t novf) {
    for (int a = 0; a < kO1Ctx; a++) {
        pi[a] = 1.0 / kO1Ctx;
        norm[a * kO1Sym + 255] = (int16_t)escape;
    }
    return split_plan(m, novf, bits, pi, (const uint8_t*)norm, false);
}
static uint64_t parts(const SplitPlan& p, uint64_t m, double bits) {
    return split_parts((int64_t)(bits * (double)m), split_sub_bits(p, bits));
}
int main() {
    int split = 0, dropped = 0, mixed = 0;
    for (uint64_t m = 8192; m <= 1ull << 28; m *= 4)
        for (double bits = 2.5; bits < 13; bits += 0.25)
            for (int esc = 1; esc < 4096; esc += esc / 8 + 1) {
                const SplitPlan p = plan(m, bits, esc, m * esc / 8192);
                if (p.cls == kSplitNone) continue;
                split++;
                // what one chain may take, and that its pool holds what was counted for such plans (0.9 from 6.5 bits
                // on, 1.2 below)
                const uint64_t ns = parts(p, m, bits);
                CHECK(split_bytes(p, m, ns) <= 80.0 * (double)m + 65536, "%g bytes a symbol", split_bytes(p, m, ns) / m)
                CHECK(split_nodes(p, m, ns) >= (bits >= 6.5 ? 0.9 : 1.2) * p.nodes * (double)m, "%g", p.nodes)
                // calls of 1 to 64 such chains, a chain decoded from its start among them or not
                for (int n = 1; n <= 64; n *= 4)
                    for (int serial = 0; serial < 2; serial++) {
                        std::vector<SplitPlan> ps(n, p);
                        std::vector<SplitCand> c;
                        for (SplitPlan& x : ps) c.push_back(SplitCand{&x, m, ns});
                        const double limit = (double)split_limit(n * m);
                        split_choose(c, limit, serial ? m : 0);
                        double total = 0, nodes = 0;
                        int left = 0;
                        for (const SplitPlan& x : ps)
                            if (x.cls != kSplitNone) {
                                total += split_bytes(x, m, ns);
                                nodes += x.nodes * (double)m;
                                left++;
                                if (serial || left < n) mixed++;
                            }
                        CHECK(total <= limit, "%g of %g, %d chains of %llu", total, limit, n, (unsigned long long)m)
                        if (!serial && n * split_bytes(p, m, ns) <= limit) CHECK(left == n, "%d of %d left", left, n)
                        if (serial || left < n) CHECK(nodes <= kSplitMixed * (double)m, "%g nodes", nodes)
                        dropped += left < n;
                    }
            }
    CHECK(split > 1000 && dropped > 100 && mixed > 1000, "%d %d %d", split, dropped, mixed)
    // the limit: no more than 64 bytes a code, a gigabyte and 4 bytes a code
    for (uint64_t n = 1; n < 1ull << 40; n *= 3) CHECK(split_limit(n) <= 64 * n && split_limit(n) <= (1ull << 30) + 4 * n, "")
    // differing chains: the most bytes a symbol go first, and what is left fits
    SplitPlan few = plan(1 << 20, 7.0, 2, 0), many = plan(1 << 20, 7.5, 200, 20000);
    CHECK(few.cls == kSplitFew && many.cls == kSplitMany, "%d %d", few.cls, many.cls)
    const uint64_t nf = parts(few, 1 << 20, 7.0), nm = parts(many, 1 << 20, 7.5);
    std::vector<SplitCand> c{{&few, 1 << 20, nf}, {&many, 1 << 20, nm}};
    split_choose(c, split_bytes(few, 1 << 20, nf) + 1000, 0);
    CHECK(few.cls == kSplitFew && many.cls == kSplitNone, "%d %d", few.cls, many.cls)
    return 0;
}
"""


def test_plans_fit_their_limit(tmp_path):
    src, exe = tmp_path / "plans.cpp", tmp_path / "plans"
    src.write_text(PLANS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "falcons_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def split_limit(n):
    return min(64 * n, (1 << 30) + 4 * n)


def workspace(n, es, pre):
    """What a decompress call reserves, every value unpredictable."""
    return n * (es + 14) + n * es + 2 * pre + (64 << 20)


def compressed(data, mode, eb):
    import falcons_amd
    cfg = falcons_amd.falconsConfig(*data.shape)
    cfg.cmprAlgo = falcons_amd.falconsAlgorithm.INTERP
    cfg.errorBoundMode = mode
    if mode:
        cfg.relErrorBound = eb
    else:
        cfg.absErrorBound = eb
    ctx = falcons_amd.Context(0)
    stream, _, _ = ctx.compress_ex(data.copy(), cfg)
    bound = ctx.prezstd_bound(cfg, data.dtype)
    ctx.close()
    return np.array(stream, dtype=np.uint8), bound


def from_the_start(ctx, stream, dtype, monkeypatch):
    monkeypatch.setenv("FALCONS_O1_SEQUENTIAL", "1")
    ref, _, _ = ctx.decompress_ex(stream, dtype)
    monkeypatch.delenv("FALCONS_O1_SEQUENTIAL")
    return ref.reshape(-1).view(np.uint8).copy()


def many_nodes():
    return (4000 + 700 * synth.power_law((101, 128, 150), -3.0, seed=1)).round().astype(np.int32), 0, 4.0


@pytest.mark.gpu
def test_held_workspace(monkeypatch, capfd):
    """A field whose graphs are large (3 nodes a code): the call holds no more than what calls are admitted by."""
    import falcons_amd
    data, mode, eb = many_nodes()
    stream, bound = compressed(data, mode, eb)
    ctx = falcons_amd.Context(0)
    want = from_the_start(ctx, stream, data.dtype, monkeypatch)
    monkeypatch.setenv("FALCONS_ARENA_STATS", "1")
    monkeypatch.setenv("FALCONS_DECODE_STATS", "1")
    capfd.readouterr()
    got, _, _ = ctx.decompress_ex(stream, data.dtype)
    err = capfd.readouterr().err
    ctx.close()
    assert np.array_equal(got.reshape(-1).view(np.uint8), want)
    assert "split chains" in err
    nodes, room = (int(x) for x in re.search(r", (\d+) nodes of (\d+)", err).groups())
    assert data.size < nodes <= room, err[-1000:]
    reserved, peak = (int(x) for x in re.search(r"\[arena\] decompress n=\d+ reserved (\d+) peak (\d+)", err).groups())
    assert peak <= reserved <= workspace(data.size, data.itemsize, bound) + split_limit(data.size), err[-1000:]


@pytest.mark.gpu
@pytest.mark.parametrize("room,split", [(0, 0), (330000, 2), (1 << 30, 4)])
def test_less_memory_than_asked_for(room, split, monkeypatch, capfd):
    """Chains that find no memory are decoded from their start, beside the split ones. Four chains of 264,000
    codes take 0.12 MB each."""
    import falcons_amd
    data = synth.power_law((1025, 1031), -3.0, seed=4)
    stream, _ = compressed(data, 1, 1e-3)
    ctx = falcons_amd.Context(0)
    want = from_the_start(ctx, stream, data.dtype, monkeypatch)
    monkeypatch.setenv("FALCONS_SIDE_BYTES", str(room))
    monkeypatch.setenv("FALCONS_DECODE_STATS", "1")
    capfd.readouterr()
    print(f"case {room} bytes", flush=True)
    got, _, _ = ctx.decompress_ex(stream, data.dtype)
    err = capfd.readouterr().err
    ctx.close()
    assert np.array_equal(got.reshape(-1).view(np.uint8), want)
    m = re.search(r"\[o1 decode\] (\d+) split chains", err)
    assert (int(m[1]) if m else 0) == split, err[-1000:]


@pytest.mark.gpu
@pytest.mark.parametrize("spare", [0, 1 << 20, 1 << 30])
def test_request_budget(spare, monkeypatch):
    """A budget that holds the request's workspace and `spare` bytes for the split decoder: served, and within it."""
    import falcons_amd
    data, mode, eb = many_nodes()
    stream, bound = compressed(data, mode, eb)
    ctx = falcons_amd.Context(0)
    want = from_the_start(ctx, stream, data.dtype, monkeypatch)
    ctx.close()
    n, es = data.size, data.itemsize
    budget = n * es + workspace(n, es, bound) + spare
    srv = falcons_amd.Server(0, slots=2, hbm_budget=budget)
    try:
        for tag in range(3):
            srv.submit_decompress(tag, stream, data.dtype, n)
        for _ in range(3):
            r = srv.poll(timeout_ms=60000)
            assert r is not None, "server stalled"
            assert r["status"] == 0, r["msg"]
            assert np.array_equal(r["out"].reshape(-1).view(np.uint8), want)
        st = srv.stats()
        assert st["completed"] == 3 and st["max_held_bytes"] <= budget and st["held_bytes"] <= budget
    finally:
        srv.close()
