"""The work that users of this library have it do, as cases that can be timed.

A case names an entry point ("kind"), a field ("field", "shape", "dtype") and a configuration
("mode", "eb", "algo"); a batched case has a chunk count instead of a shape. The fields are the
workloads of bench.py and the tests (falcons_amd/synth.py), synthesised on the GPU:

  power   Gaussian random field with power spectrum |k|^-3, zero mean and unit variance, a crop of a
          periodic field whose sides are powers of two
  front   |k|^-5/3 field plus a smooth radial tanh front of width 8 cells
  waves   16 sinusoids of integer frequency 1..8 per axis plus N(0, 1e-3) noise
  counts  the power field scaled to integers of some thousands (detector counts, stored as int32)

kinds:
  compress          Context.compress_device on a field in HBM. The call overwrites its input with the
                    reconstruction, so a pass first copies the field to the buffer that the call takes.
  decompress        Context.decompress_device into HBM
  roundtrip         both, one after the other
  batch_compress    Context.compress_batch over uneven chunks
  batch_decompress  Context.decompress_batch over uneven chunks
  host              falcons.compress and falcons.decompress on numpy arrays (zstd and transfers included)
"""
import math
import random

import numpy as np
import torch

import falcons_amd as fa

_DEVICE = "cuda"
_MODES = {"abs": fa.falconsErrorBoundMode.ABS, "rel": fa.falconsErrorBoundMode.REL}
_ALGOS = {"interp": fa.falconsAlgorithm.INTERP, "search": fa.falconsAlgorithm.INTERP_LORENZO}
_TORCH = {"float32": torch.float32, "float64": torch.float64, "int32": torch.int32}
_CHUNK_RELS = (1e-2, 1e-3, 1e-4)


def listed():
    def case(name, kind, shape, eb, mode="rel", field="power", dtype="float32", algo="interp"):
        return {"name": name, "kind": kind, "shape": "x".join(str(s) for s in shape), "field": field, "dtype": dtype,
                "mode": mode, "eb": eb, "algo": algo}

    def batch(name, kind, chunks):
        return {"name": name, "kind": kind, "chunks": chunks}

    cube = (512, 512, 512)
    return [
        # one small variable of a simulation's output step, written and read back on its own: launches
        # and host round trips
        case("small_roundtrip", "roundtrip", (33, 40, 65), 1e-3),
        # the uneven blocks of an adaptive mesh, many to a call
        batch("chunks_compress", "batch_compress", 48),
        batch("chunks_decompress", "batch_decompress", 192),
        # an integer dataset's chunk (HDF5 integer types), the generic traversal
        case("counts_roundtrip", "roundtrip", (101, 128, 150), 4.0, mode="abs", field="counts", dtype="int32"),
        # the library called as pyfalcons is, arrays in host memory, zstd frame included
        case("host_roundtrip", "host", (128, 128, 128), 1e-3, mode="abs", field="waves"),
        # an image or climate plane with odd sides, read back
        case("plane_decompress", "decompress", (3001, 2047), 1e-3),
        # double precision snapshot with a front, tight absolute bound, parameters searched per call
        case("front_f64_compress", "compress", (256, 384, 384), 1e-6, mode="abs", field="front", dtype="float64",
             algo="search"),
        case("front_f64_decompress", "decompress", (256, 384, 384), 1e-6, mode="abs", field="front",
             dtype="float64", algo="search"),
        # the benchmark's field at its two bounds, each direction on its own
        case("cube_compress_1e-3", "compress", cube, 1e-3),
        case("cube_decompress_1e-3", "decompress", cube, 1e-3),
        case("cube_compress_1e-4", "compress", cube, 1e-4),
        case("cube_decompress_1e-4", "decompress", cube, 1e-4),
    ]


def draw(rng):
    """One more case: entry point by how often programs use it, sides log-uniform (odd ones as they
    come), bounds log-uniform from 1e-4 to 1e-2 of the range."""
    kind = rng.choice(["compress", "compress", "decompress", "decompress", "roundtrip", "host", "batch_compress",
                       "batch_decompress"])
    if kind == "batch_compress":
        return {"kind": kind, "chunks": rng.randint(8, 56)}
    if kind == "batch_decompress":
        return {"kind": kind, "chunks": rng.randint(8, 192)}
    field, dtype = rng.choice([("power", "float32")] * 5 + [("waves", "float32"), ("power", "float64"),
                                                            ("front", "float64"), ("counts", "int32")])
    ndim = 3 if field in ("front", "counts") else rng.choice([1, 2, 2, 3, 3, 3, 3])
    lo, hi = {1: (1 << 14, 1 << 22), 2: (128, 3072), 3: (32, 400)}[ndim]
    if kind in ("roundtrip", "host"):  # smaller fields: a variable or a chunk at a time
        hi = {1: 1 << 20, 2: 1024, 3: 128}[ndim]
    if dtype != "float32":
        hi = hi * 3 // 4
    shape = [int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) for _ in range(ndim)]
    if field == "counts":
        mode, eb, algo = "abs", float(rng.randint(1, 16)), "interp"
    else:
        mode, eb = "rel", float("%.3g" % 10 ** rng.uniform(-4, -2))
        algo = "search" if dtype == "float64" and ndim > 1 and rng.random() < 0.5 else "interp"
    return {"kind": kind, "shape": "x".join(str(s) for s in shape), "field": field, "dtype": dtype, "mode": mode,
            "eb": eb, "algo": algo}


def _shape(case):
    return tuple(int(s) for s in case["shape"].split("x"))


def _spectral(shape, slope, gen, dtype):
    """A random field of power spectrum |k|^slope: a crop of a periodic one with power-of-two sides."""
    full = [1 << max(3, (s - 1).bit_length()) for s in shape]
    spec = torch.fft.rfftn(torch.randn(full, generator=gen, device=_DEVICE, dtype=dtype))
    k2 = torch.zeros((), device=_DEVICE, dtype=dtype)
    for i, n in enumerate(full):
        freq = torch.fft.rfftfreq if i == len(full) - 1 else torch.fft.fftfreq
        k2 = k2 + (freq(n, device=_DEVICE, dtype=dtype) ** 2).reshape([-1 if j == i else 1 for j in range(len(full))])
    k2.view(-1)[0] = 1.0
    amp = k2 ** (slope / 4.0)
    amp.view(-1)[0] = 0.0
    spec *= amp
    del amp, k2
    f = torch.fft.irfftn(spec, s=full)[tuple(slice(0, s) for s in shape)].contiguous()
    f -= f.mean()
    return f / f.std()


def _field(case, seed):
    shape, dtype = _shape(case), _TORCH[case["dtype"]]
    gen = torch.Generator(device=_DEVICE).manual_seed(seed)
    if case["field"] == "power":
        return _spectral(shape, -3.0, gen, dtype)
    if case["field"] == "counts":
        return (4000.0 + 700.0 * _spectral(shape, -3.0, gen, torch.float32)).round().to(torch.int32)
    if case["field"] == "front":
        f = _spectral(shape, -5.0 / 3.0, gen, dtype)
        r2 = torch.zeros((), device=_DEVICE, dtype=dtype)
        for i, s in enumerate(shape):
            g = torch.arange(s, device=_DEVICE, dtype=dtype) - (s - 1) / 2
            r2 = r2 + (g * g).reshape([-1 if j == i else 1 for j in range(len(shape))])
        return f + torch.tanh((r2.sqrt() - 0.3 * min(shape)) / 8.0)
    rng = random.Random(seed)  # waves
    f = 1e-3 * torch.randn(shape, generator=gen, device=_DEVICE, dtype=torch.float64)
    for _ in range(16):
        amp, phase = rng.uniform(0.1, 1.0), rng.uniform(0.0, 2 * math.pi)
        arg = torch.full((), phase, device=_DEVICE, dtype=torch.float64)
        for i, s in enumerate(shape):
            x = torch.arange(s, device=_DEVICE, dtype=torch.float64) * (2 * math.pi * rng.randint(1, 8) / s)
            arg = arg + x.reshape([-1 if j == i else 1 for j in range(len(shape))])
        f += amp * torch.sin(arg)
    return f.to(dtype)


def _config(shape, mode, eb, algo="interp"):
    cfg = fa.falconsConfig(*shape)
    cfg.cmprAlgo = _ALGOS[algo]
    cfg.errorBoundMode = _MODES[mode]
    if mode == "abs":
        cfg.absErrorBound = eb
    else:
        cfg.relErrorBound = eb
    return cfg


class _Buffer:
    """A tensor in HBM where the Context methods take a device buffer."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.nbytes = tensor, tensor.data_ptr(), tensor.numel() * tensor.element_size()


def _chunks(case, seed):
    """Sides and relative bound of each chunk (the mesh stays as it is), and the chunks themselves: crops
    of one |k|^-3 field at places of the mesh, one after another in a flat tensor (256-byte aligned)."""
    rng = random.Random(case["chunks"])
    base = _spectral((256, 256, 256), -3.0, torch.Generator(device=_DEVICE).manual_seed(seed), torch.float32)
    plan, parts = [], []
    for _ in range(case["chunks"]):
        shape = [int(math.exp(rng.uniform(math.log(32), math.log(128)))) for _ in range(3)]
        at = [rng.randint(0, 256 - s) for s in shape]
        part = base[tuple(slice(o, o + s) for o, s in zip(at, shape))].reshape(-1)
        plan.append((tuple(shape), rng.choice(_CHUNK_RELS), sum(p.numel() for p in parts)))
        parts.append(torch.nn.functional.pad(part, (0, -part.numel() % 64)))
    return plan, torch.cat(parts)


def _store_bytes(n, size):
    """Room that a program sets aside to store the stream of a field of n values: the streams of these
    cases are shorter than their fields, those of the smallest by no more than some tables."""
    return n * size + (1 << 17)


_context = None


def _ctx():
    """A program keeps one context."""
    global _context
    if _context is None:
        _context = fa.Context(0)
    return _context


def _compressed(ctx, cfg, dtype, field):
    """What a program has in hand that reads a stored field: the stream in HBM, its host copy (the
    headers are parsed from it) and the stream's configuration."""
    cfg = cfg.copy()
    pre = torch.empty(ctx.prezstd_bound(cfg, dtype), dtype=torch.uint8, device=_DEVICE)
    work = field.clone()
    torch.cuda.synchronize()
    n, _ = ctx.compress_device(cfg, dtype, _Buffer(work), _Buffer(pre))
    pre = pre[:n].clone()
    return cfg, pre, pre.cpu().numpy()


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    state = {"ctx": ctx, "kind": kind}
    if kind.startswith("batch"):
        plan, fields = _chunks(case, seed)
        state["orig"], state["work"] = fields, torch.empty_like(fields)
        state["items"] = items = []
        if kind == "batch_compress":
            rooms = [_store_bytes(math.prod(shape), 4) for shape, _, _ in plan]
            state["store"] = torch.zeros(sum(rooms), dtype=torch.uint8, device=_DEVICE)
            state["stores"] = torch.split(state["store"], rooms)
        for shape, rel, at in plan:
            n = math.prod(shape)
            cfg = _config(shape, "rel", rel)
            if kind == "batch_compress":
                pre = torch.empty(ctx.prezstd_bound(cfg, np.float32), dtype=torch.uint8, device=_DEVICE)
                items.append((cfg, np.float32, _Buffer(state["work"][at:at + n]), _Buffer(pre)))
            else:
                cfg, pre, h_pre = _compressed(ctx, cfg, np.float32, fields[at:at + n])
                items.append((cfg, np.float32, h_pre, _Buffer(pre), _Buffer(state["work"][at:at + n])))
        if kind == "batch_decompress":
            state["work"].zero_()
        torch.cuda.synchronize()
        return state
    dtype = np.dtype(case["dtype"])
    field = _field(case, seed)
    cfg = _config(_shape(case), case["mode"], case["eb"], case["algo"])
    state.update(cfg=cfg, dtype=dtype, shape=_shape(case))
    room = _store_bytes(field.numel(), dtype.itemsize)
    if kind == "host":
        state["data"], state["store"] = field.cpu().numpy(), np.zeros(room, dtype=np.uint8)
        return state
    if kind != "compress":
        state["stream"] = _compressed(ctx, cfg, dtype, field)
        state["out"] = _Buffer(torch.empty_like(field))
    if kind != "decompress":
        state["orig"] = field
        state["work"] = _Buffer(torch.empty_like(field))
        state["pre"] = _Buffer(torch.empty(ctx.prezstd_bound(cfg, dtype), dtype=torch.uint8, device=_DEVICE))
        state["store"] = torch.zeros(room, dtype=torch.uint8, device=_DEVICE)
    torch.cuda.synchronize()
    return state


def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind == "batch_compress":
        state["work"].copy_(state["orig"])
        torch.cuda.current_stream().synchronize()  # the library's streams do not wait for torch's
        items = [(cfg.copy(), dtype, data, pre) for cfg, dtype, data, pre in state["items"]]
        sizes, _, _ = ctx.compress_batch(items)
        for (_, _, _, pre), n, store in zip(items, sizes, state["stores"]):
            store[:n].copy_(pre.tensor[:n])
        return {"sizes": np.array(sizes), "streams": state["store"], "fields": state["work"]}
    if kind == "batch_decompress":
        ctx.decompress_batch(state["items"])
        return {"fields": state["work"]}
    if kind == "host":
        stream, _ = fa.falcons.compress(state["data"], state["cfg"].copy(), copy=True)
        state["store"][:stream.size] = stream
        field, _ = fa.falcons.decompress(stream, state["dtype"], state["shape"])
        return {"size": int(stream.size), "stream": state["store"], "field": field}
    got = {}
    if kind != "decompress":
        state["work"].tensor.copy_(state["orig"])
        torch.cuda.current_stream().synchronize()
        n, _ = ctx.compress_device(state["cfg"].copy(), state["dtype"], state["work"], state["pre"])
        state["store"][:n].copy_(state["pre"].tensor[:n])  # out of the call's large buffer, to be kept
        got["size"], got["stream"], got["reconstruction"] = int(n), state["store"], state["work"].tensor
    if kind != "compress":
        cfg, pre, h_pre = state["stream"]
        ctx.decompress_device(cfg, state["dtype"], h_pre, _Buffer(pre), state["out"])
        got["field"] = state["out"].tensor
    return got


def work(case):
    """Field and stream read or written once each. Stream sizes follow from the bound: about 2.2 bits a
    value at 1e-2 of the range, 6.3 at 1e-3 and 9.7 at 1e-4 (measured on the 512^3 field); the other
    fields' bounds are taken as their share of a range of about 8 standard deviations."""
    def bits(share):
        return min(24.0, max(0.5, 6.3 + 3.5 * math.log10(1e-3 / share)))

    kind = case["kind"]
    if kind.startswith("batch"):
        n = case["chunks"] * ((128 - 32) / math.log(4)) ** 3
        stream, size, ways = n * 6.1 / 8, 4, (2 if kind == "batch_compress" else 1)
        return {"bytes": n * size * ways + stream, "flops": 0}
    n, size = math.prod(_shape(case)), np.dtype(case["dtype"]).itemsize
    share = case["eb"]
    if case["mode"] == "abs":
        share = share / (5600.0 if case["field"] == "counts" else 8.0)
    stream = n * bits(share) / 8
    compress, decompress = 2 * n * size + stream, n * size + stream
    return {"bytes": {"compress": compress, "decompress": decompress}.get(kind, compress + decompress), "flops": 0}


def exact(case, seed):
    """The field itself, in 64 bits: what every reconstruction and decompressed field approximates
    within the case's bound. Streams are bytes, and an integer field stays as it is."""
    kind = case["kind"]
    if kind.startswith("batch"):
        fields = _chunks(case, seed)[1].double()
        return {"sizes": None, "streams": None, "fields": fields} if kind == "batch_compress" else {"fields": fields}
    if case["dtype"] == "int32":
        return None
    field = _field(case, seed).double()
    if kind == "host":
        return {"size": None, "stream": None, "field": field.cpu().numpy()}
    got = {}
    if kind != "decompress":
        got["size"], got["stream"], got["reconstruction"] = None, None, field
    if kind != "compress":
        got["field"] = field
    return got
