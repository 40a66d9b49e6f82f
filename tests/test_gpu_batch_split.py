"""Split order-1 chains of many fields in one set of launches: every field of a batch must equal, bit for bit,
what a plain call that decodes every chain from its first symbol gives; fields of each size class of the
split decoder's graphs, beside fields whose chains are too short or too rich in escapes for it."""
import numpy as np
import pytest

from falcons_amd import synth

pytestmark = pytest.mark.gpu

# shape, bound; a chain holds a quarter of the codes (8,192 at least to be split)
FIELDS = [((33, 40, 65), 1e-3), ((60, 71, 82), 1e-2), ((60, 71, 82), 1e-3), ((60, 71, 82), 1e-4), ((101, 102, 103), 1e-2),
          ((150001,), 1e-3), ((1025, 1031), 1e-3), ((81, 64, 75), 7e-4), ((20, 21, 22), 1e-4), ((33, 31, 32), 1e-3)]


@pytest.mark.parametrize("workers,times", [(1, 1), (4, 3)])
def test_batch_of_split_chains(monkeypatch, workers, times):
    import falcons_amd
    ctx = falcons_amd.Context(0)
    items, refs, bufs = [], [], []
    for k, (shape, eb) in enumerate(FIELDS * times):
        dtype = np.float64 if k % 4 == 3 else np.float32
        data = synth.power_law(shape, -3.0 if len(shape) > 1 else -2.0, seed=30 + k, dtype=dtype)
        cfg = falcons_amd.falconsConfig(*shape)
        cfg.cmprAlgo = falcons_amd.falconsAlgorithm.INTERP
        cfg.errorBoundMode = 1
        cfg.relErrorBound = eb
        d, p = ctx.alloc(data.nbytes), ctx.alloc(ctx.prezstd_bound(cfg, dtype))
        d.upload(data)
        n, _ = ctx.compress_device(cfg, dtype, d, p)
        pre = p.download(n)
        ref, o = ctx.alloc(data.nbytes), ctx.alloc(data.nbytes)
        monkeypatch.setenv("FALCONS_O1_SEQUENTIAL", "1")
        ctx.decompress_device(cfg, dtype, pre, None, ref)
        monkeypatch.delenv("FALCONS_O1_SEQUENTIAL")
        refs.append(ref.download(data.nbytes, dtype))
        items.append((cfg, dtype, pre, p if k % 2 else None, o))
        bufs += [d, p, ref, o]
    ctx.set_workers(workers)
    print(f"case {workers} workers, {len(items)} fields", flush=True)
    for _ in range(2):
        status, _ = ctx.decompress_batch(items)
        assert status == [0] * len(items)
        for (cfg, dtype, _, _, o), ref in zip(items, refs):
            assert np.array_equal(o.download(ref.nbytes, dtype).view(np.uint8), ref.view(np.uint8))
    for b in bufs:
        b.free()
    ctx.close()
