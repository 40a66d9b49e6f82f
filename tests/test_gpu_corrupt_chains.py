"""Damaged bits in the body of an order-1 tANS chain, whose framing is whole: nothing in the format tells, so a call may
end in an error or in another field, but it ends, it does the same whenever it is made, the two decoders agree
where both give a field, and the next call is none the worse."""
import struct

import numpy as np
import pytest

from falcons_amd import synth

pytestmark = pytest.mark.gpu

FIELDS = {
    "few": lambda: (synth.power_law((513, 515), -3.0, seed=4), 1e-3),
    "some": lambda: (synth.power_law((61, 70, 83), -3.0, seed=5), 1e-3),
    "many": lambda: (synth.power_law((90, 67, 71), -3.0, seed=6, dtype=np.float64), 7e-4),
}


def chains_of(pre):
    """(offset, length) of the four chains of a one-segment order-1 stream in a pre-zstd buffer."""
    b = pre.tobytes()
    at = -1
    while True:
        at = b.find(struct.pack("<Q", 1), at + 1)
        assert at >= 0
        n, k = struct.unpack_from("<QQ", b, at + 8)
        if k != 4 or not 1000 < n < 1 << 23:
            continue
        blen = struct.unpack_from("<4Q", b, at + 24)
        body = at + 24 + 64 + 15 * 256 * 2
        if body + sum(blen) <= len(b) and all(1000 < x for x in blen):
            return [(body + sum(blen[:q]), blen[q]) for q in range(4)]


def damages(rng, pre):
    for q, (off, size) in enumerate(chains_of(pre)):
        for where in (0.02, 0.5, 0.97):
            at = off + int(size * where)
            bad = pre.copy()
            bad[at] ^= 1 << int(rng.integers(8))
            yield f"bit in chain {q} at {where}", bad
        for what in ("zeros", "ones", "noise"):
            w = int(rng.integers(100, size // 2))
            at = off + int(rng.integers(0, size - w - 8))
            bad = pre.copy()
            bad[at:at + w] = {"zeros": 0, "ones": 255}.get(what, rng.integers(0, 256, w))
            yield f"{what} in chain {q}", bad


@pytest.mark.parametrize("name", list(FIELDS))
def test_damaged_chain_bodies(name, monkeypatch):
    import falcons_amd
    ctx = falcons_amd.Context(0)
    data, eb = FIELDS[name]()
    cfg = falcons_amd.falconsConfig(*data.shape)
    cfg.cmprAlgo = falcons_amd.falconsAlgorithm.INTERP
    cfg.errorBoundMode = 1
    cfg.relErrorBound = eb
    d, p, o = ctx.alloc(data.nbytes), ctx.alloc(ctx.prezstd_bound(cfg, data.dtype)), ctx.alloc(data.nbytes)
    d.upload(data)
    n, _ = ctx.compress_device(cfg, data.dtype, d, p)
    pre = p.download(n)

    def decode(buf):
        try:
            ctx.decompress_device(cfg, data.dtype, buf, None, o)
        except (ValueError, falcons_amd.FalconsError) as e:
            return str(e)
        return o.download(data.nbytes, data.dtype).view(np.uint8)

    whole = decode(pre)
    assert not isinstance(whole, str)
    errors = 0
    for what, bad in damages(np.random.default_rng(3), pre):
        print(f"case {name}: {what}", flush=True)
        monkeypatch.delenv("FALCONS_O1_SEQUENTIAL", raising=False)
        monkeypatch.setenv("FALCONS_O1_PARALLEL_SHORT", "1")
        split, again = decode(bad), decode(bad)
        monkeypatch.setenv("FALCONS_O1_SEQUENTIAL", "1")
        start = decode(bad)
        assert type(split) is type(again) and np.array_equal(split, again)
        if not isinstance(split, str) and not isinstance(start, str):
            assert np.array_equal(split, start)
        errors += isinstance(split, str)
    assert errors > 0
    monkeypatch.delenv("FALCONS_O1_SEQUENTIAL")
    assert np.array_equal(decode(pre), whole)
    for b in (d, p, o):
        b.free()
    ctx.close()
