"""Batched decompress with less device memory for its split order-1 chains than they ask for: none at all (the
shared launch fails and every item goes through a plain call), or a part (the other chains are decoded from
their start). Every field equals that of plain calls which decode every chain from its first symbol."""
import numpy as np
import pytest

from falcons_amd import synth

pytestmark = pytest.mark.gpu

# the last one's chains are longer than a batch takes by itself, and need more than its item's region has room for
FIELDS = [((33, 40, 65), 1e-3), ((60, 71, 82), 1e-2), ((60, 71, 82), 1e-4), ((1025, 1031), 1e-3), ((20, 21, 22), 1e-4),
          ((160, 160, 160), 6e-4)]


@pytest.fixture(scope="module")
def batch():
    import falcons_amd
    mp = pytest.MonkeyPatch()
    ctx = falcons_amd.Context(0)
    items, refs, bufs = [], [], []
    for k, (shape, eb) in enumerate(FIELDS):
        data = synth.power_law(shape, -3.0, seed=50 + k)
        cfg = falcons_amd.falconsConfig(*shape)
        cfg.cmprAlgo = falcons_amd.falconsAlgorithm.INTERP
        cfg.errorBoundMode = 1
        cfg.relErrorBound = eb
        d, p = ctx.alloc(data.nbytes), ctx.alloc(ctx.prezstd_bound(cfg, data.dtype))
        d.upload(data)
        n, _ = ctx.compress_device(cfg, data.dtype, d, p)
        pre = p.download(n)
        ref, o = ctx.alloc(data.nbytes), ctx.alloc(data.nbytes)
        mp.setenv("FALCONS_O1_SEQUENTIAL", "1")
        ctx.decompress_device(cfg, data.dtype, pre, None, ref)
        mp.delenv("FALCONS_O1_SEQUENTIAL")
        refs.append(ref.download(data.nbytes, data.dtype))
        items.append((cfg, data.dtype, pre, p, o))
        bufs += [d, p, ref, o]
    ctx.set_workers(3)
    yield ctx, items, refs
    for b in bufs:
        b.free()
    ctx.close()


@pytest.mark.parametrize("switch,room", [(None, 0), ("FALCONS_SIDE_BYTES", 0), ("FALCONS_SIDE_BYTES", 300000),
                                         ("FALCONS_BATCH_SPLIT_BYTES", 0), ("FALCONS_BATCH_SPLIT_BYTES", 400000)])
def test_batch_with_less_memory(batch, monkeypatch, switch, room):
    ctx, items, refs = batch
    if switch:
        monkeypatch.setenv(switch, str(room))
    print(f"case {switch} {room}", flush=True)
    for _ in range(2):
        for (_, dtype, _, _, o), ref in zip(items, refs):
            o.upload(np.zeros_like(ref))
        status, _ = ctx.decompress_batch(items)
        assert status == [0] * len(items)
        for (_, dtype, _, _, o), ref in zip(items, refs):
            assert np.array_equal(o.download(ref.nbytes, dtype).view(np.uint8), ref.view(np.uint8))
