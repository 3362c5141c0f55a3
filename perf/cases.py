"""Timed cases: what a program that uses prism_amd has it do.

A program compresses a field that is in device memory (pipeline.compress),
decompresses a plain stream whole (pipeline.decompress), refines a
progressive stream through a series of bounds (pipeline.Retriever), or does
the first and the last for many small fields at once
(pipeline.BatchCompressor, pipeline.retrieve_batch).  The fields are 1-D, 2-D
and 3-D, float32 and float64, from a 64^3 block to a 512^3 cube, with bounds
from 1e-2 to 1e-6 of the value range.
"""
import math

import numpy as np
import torch

from prism_amd import fields, pipeline

DT = {"f32": torch.float32, "f64": torch.float64}
ITEM = {"f32": 4, "f64": 8}
MOST_BYTES = 512 * 512 * 512 * 4  # the largest field of the range


def listed():
    return [
        # The smallest call in earnest: one 64^3 block of a simulation, written
        # out with a plain (non-progressive) stream.  Launches and host time.
        {"name": "compress_64_f32", "kind": "compress", "nx": 64, "ny": 64, "nz": 64, "dtype": "f32",
         "field": "mix", "eb": 1e-3, "rel": True, "progressive": False},
        # ... and read back whole.
        {"name": "decompress_64_f32", "kind": "decompress", "nx": 64, "ny": 64, "nz": 64, "dtype": "f32",
         "field": "mix", "eb": 1e-3, "rel": True, "progressive": False},
        # The usual snapshot: a hydrodynamics density field in double precision,
        # archived once as a progressive stream at a tight bound.
        {"name": "compress_density_f64", "kind": "compress", "nx": 384, "ny": 384, "nz": 256, "dtype": "f64",
         "field": "density", "eb": 1e-6, "rel": True, "progressive": True},
        # ... and looked at: a rough view first, refined a decade at a time.
        {"name": "retrieve_density_f64", "kind": "retrieve", "nx": 384, "ny": 384, "nz": 256, "dtype": "f64",
         "field": "density", "eb": 1e-6, "rel": True, "progressive": True, "first": 1e-2, "rounds": 5},
        # The largest: a 512^3 turbulence-like cube in single precision, whose
        # codes keep many more bits than the smooth fields' do.
        {"name": "compress_grf512_f32", "kind": "compress", "nx": 512, "ny": 512, "nz": 512, "dtype": "f32",
         "field": "grf", "eb": 1e-4, "rel": True, "progressive": True},
        {"name": "retrieve_grf512_f32", "kind": "retrieve", "nx": 512, "ny": 512, "nz": 512, "dtype": "f32",
         "field": "grf", "eb": 1e-4, "rel": True, "progressive": True, "first": 1e-1, "rounds": 4},
        # A checkpoint on a grid whose axes are no multiples of anything,
        # restored whole.
        {"name": "decompress_ragged_f64", "kind": "decompress", "nx": 301, "ny": 257, "nz": 385, "dtype": "f64",
         "field": "density", "eb": 1e-5, "rel": True, "progressive": False},
        # A 2-D map, compressed under an absolute bound (what a program does
        # that knows its instrument's accuracy).
        {"name": "compress_map_f64", "kind": "compress", "nx": 1999, "ny": 1801, "nz": 1, "dtype": "f64",
         "field": "modes", "eb": 1e-3, "rel": False, "progressive": False},
        # A long 1-D series (a flattened field, a particle coordinate).
        {"name": "compress_series_f32", "kind": "compress", "nx": 6000001, "ny": 1, "nz": 1, "dtype": "f32",
         "field": "modes", "eb": 1e-4, "rel": True, "progressive": True},
        # A 2-D map refined interactively: each round is short, and its
        # latency is what the viewer waits for.
        {"name": "retrieve_map_f32", "kind": "retrieve", "nx": 1388, "ny": 1679, "nz": 1, "dtype": "f32",
         "field": "density", "eb": 1e-5, "rel": True, "progressive": True, "first": 1e-2, "rounds": 3},
        # All 64 variables of a time step, mixed shapes and types, through one
        # plan that is kept for the whole run; each step brings new fields.
        {"name": "batch64_compress", "kind": "batch_compress", "fields": 64, "spec": 100},
        # 16 resident fields, each refined in every batch of a serving loop.
        {"name": "batch16_retrieve", "kind": "batch_retrieve", "fields": 16, "spec": 100, "first": 1e-2, "rounds": 4},
    ]


def draw(rng):
    most = max(work(c)["bytes"] for c in listed())
    while True:
        c = _draw(rng)
        if c["kind"].startswith("batch"):
            n = sum(math.prod(_spec(c, i)[0]) * ITEM[_spec(c, i)[1]] for i in range(c["fields"]))
            if n > 2 * MOST_BYTES:
                continue
        elif math.prod((c["nx"], c["ny"], c["nz"])) * ITEM[c["dtype"]] > MOST_BYTES:
            continue
        if work(c)["bytes"] <= most:
            return c


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["compress"] * 6 + ["retrieve"] * 6 + ["decompress"] * 4 + ["batch_compress"] * 2 +
                      ["batch_retrieve"] * 2)
    if kind == "batch_compress":
        return {"kind": kind, "fields": _log(rng, 4, 64), "spec": rng.randint(1, 10 ** 6)}
    if kind == "batch_retrieve":
        return {"kind": kind, "fields": _log(rng, 2, 16), "spec": rng.randint(1, 10 ** 6),
                "first": 10.0 ** -rng.randint(1, 3), "rounds": rng.randint(1, 4)}
    dims = rng.choice([3, 3, 3, 3, 2, 1])
    if dims == 3:
        nx, ny, nz = _log(rng, 33, 512), _log(rng, 33, 512), _log(rng, 33, 512)
    elif dims == 2:
        nx, ny, nz = _log(rng, 64, 4096), _log(rng, 64, 4096), 1
    else:
        nx, ny, nz = _log(rng, 10 ** 5, 10 ** 7), 1, 1
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "dtype": rng.choice(["f32", "f64"]),
         "field": rng.choice(["mix", "density", "grf"] if dims == 3 else ["density", "modes"]),
         "eb": 10.0 ** rng.uniform(-6, -2), "rel": rng.random() < 0.75, "progressive": True}
    if not c["rel"]:
        c["eb"] *= 4.0  # the fields' ranges are 1 to 12
    if kind == "retrieve":
        c["first"] = 10.0 ** -rng.randint(1, 3)
        c["rounds"] = rng.randint(1, 5)
    elif kind == "decompress":
        c["progressive"] = False
    else:
        c["progressive"] = rng.random() < 0.7
    return c


# ------------------------------------------------------------------ inputs --
def _waves(shape, g, kmax, count, amp, dev):
    """Sum of `count` random-phase plane waves on [nz][ny][nx], in float64."""
    nz, ny, nx = shape
    z = torch.arange(nz, dtype=torch.float64, device=dev).view(nz, 1, 1) / nz
    y = torch.arange(ny, dtype=torch.float64, device=dev).view(1, ny, 1) / ny
    x = torch.arange(nx, dtype=torch.float64, device=dev).view(1, 1, nx) / nx
    f = torch.zeros(shape, dtype=torch.float64, device=dev)
    for _ in range(count):
        k = [int(v) if n > 1 else 0 for v, n in zip(g.randint(1, kmax + 1, 3), (nx, ny, nz))]
        ph = 2 * math.pi * g.uniform()
        a = amp(math.sqrt(sum(v * v for v in k) or 1))
        f += a * torch.sin(2 * math.pi * (k[0] * x + k[1] * y + k[2] * z) + ph)
    return f


def _field(kind, shape, dtype, seed, dev="cuda"):
    """One field: "mix" (plane waves, Gaussian blobs and a little noise),
    "density" (fronts between two plateaus and noise), "grf" (a power-law
    Gaussian random cube) or "modes" (its cheap form for 1-D and 2-D)."""
    g = np.random.RandomState(seed % (1 << 32))
    t = torch.Generator(device=dev)
    t.manual_seed(seed)
    nz, ny, nx = shape

    def noise(sigma):
        return torch.randn(shape, generator=t, dtype=torch.float64, device=dev) * sigma

    if kind == "mix":
        f = _waves(shape, g, 6, 8, lambda k: 1.0, dev)
        z = torch.arange(nz, dtype=torch.float64, device=dev).view(nz, 1, 1)
        y = torch.arange(ny, dtype=torch.float64, device=dev).view(1, ny, 1)
        x = torch.arange(nx, dtype=torch.float64, device=dev).view(1, 1, nx)
        for _ in range(4):
            a, s = 0.5 + 1.5 * g.uniform(), 4 + 6 * g.uniform()
            c = g.uniform(size=3) * (nx, ny, nz)
            f += a * torch.exp(-((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) / (2 * s * s))
        f += noise(1e-3)
    elif kind == "density":
        f = 1 + 0.5 * torch.tanh(_waves(shape, g, 8, 8, lambda k: 1.0, dev)) + noise(1e-4)
    elif kind == "grf":
        kz = torch.fft.fftfreq(nz, device=dev, dtype=torch.float64).view(nz, 1, 1) * nz
        ky = torch.fft.fftfreq(ny, device=dev, dtype=torch.float64).view(1, ny, 1) * ny
        kx = torch.fft.rfftfreq(nx, device=dev, dtype=torch.float64).view(1, 1, nx // 2 + 1) * nx
        k2 = kx * kx + ky * ky + kz * kz
        amp = torch.where(k2 > 0, k2.clamp_min(1e-30) ** (-5.0 / 12.0), torch.zeros_like(k2))
        del k2
        ph = torch.rand(amp.shape, generator=t, dtype=torch.float64, device=dev) * (2 * math.pi)
        f = torch.fft.irfftn(torch.polar(amp, ph), s=(nz, ny, nx))
        del amp, ph
        f = (f - f.mean()) / f.std()
    else:
        f = _waves(shape, g, 40, 48, lambda k: k ** (-5.0 / 6.0), dev) + noise(1e-3)
    return f.to(dtype)


def _spec(case, i):
    """Shape, type and bound of field i of a batch: the mixed batch of
    prism_amd.fields (3-D axes 32..256, 2-D axes 64..2048, 1-D 1e5..1e7)."""
    (nx, ny, nz), dtype, gen, eb = fields.batch_spec(i, case["spec"] + i)
    kind = "density" if gen == "density" else ("grf" if nz > 1 else "modes")
    return (nz, ny, nx), ("f32" if dtype == torch.float32 else "f64"), kind, eb


def _inputs(case, seed):
    """(fields, bounds) of a case"""
    if case["kind"].startswith("batch"):
        parts = [_spec(case, i) for i in range(case["fields"])]
        fs = [_field(kind, shape, DT[dt], seed * 1000 + i) for i, (shape, dt, kind, _) in enumerate(parts)]
        return fs, [eb for _, _, _, eb in parts]
    f = _field(case["field"], (case["nz"], case["ny"], case["nx"]), DT[case["dtype"]], seed)
    return [f], [case["eb"]]


def _targets(case, eb, rel):
    """The bounds of the rounds: from `first`, a decade at a time, no finer
    than the stream's own bound."""
    scale = 1.0 if rel else 4.0
    return [max(case["first"] * scale * 10.0 ** -k, eb) for k in range(case["rounds"])]


def prepare(case, seed):
    fs, ebs = _inputs(case, seed)
    s = {"case": case}
    if case["kind"] == "compress":
        s["field"], s["eb"] = fs[0], ebs[0]
        # the program's own place for the stream: the codes' 4 bytes a value
        # at most, a 1-D field's anchors and tables
        s["slot"] = torch.zeros(5 * fs[0].numel() + (1 << 19), dtype=torch.uint8, device="cuda")
    elif case["kind"] == "batch_compress":
        s["fields"], s["ebs"] = fs, ebs
        s["plan"] = pipeline.BatchCompressor(fs, ebs, rel=True, progressive=True, graph=True)
        s["plan"].outbuf.zero_()  # the streams' places, of fixed size, are compared whole
    elif case["kind"] == "batch_retrieve":
        s["streams"] = [pipeline.compress(f, eb, rel=True, progressive=True) for f, eb in zip(fs, ebs)]
        s["targets"] = [_targets(case, eb, True) for eb in ebs]
    else:
        s["stream"] = pipeline.compress(fs[0], ebs[0], rel=case["rel"], progressive=case["progressive"])
        if case["kind"] == "retrieve":
            s["targets"] = _targets(case, ebs[0], case["rel"])
    if "streams" in s or "stream" in s:  # a stream as it is loaded: of its own length, not a view of the encoder's buffer
        for c in s.get("streams", [s.get("stream")]):
            c.stream = c.stream.clone()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "compress":
        # the stream that comes back is a view of a buffer of the worst
        # case's size; a program that keeps it moves it to where it is kept
        c = pipeline.compress(s["field"], s["eb"], rel=case["rel"], progressive=case["progressive"])
        s["slot"][:c.nbytes].copy_(c.stream)
        return [s["slot"], c.nbytes]
    if kind == "decompress":
        return pipeline.decompress(s["stream"])
    if kind == "retrieve":
        r = pipeline.Retriever(s["stream"])
        return [r.retrieve(t) for t in s["targets"]]
    if kind == "batch_compress":
        cs = s["plan"].run(s["fields"], s["ebs"])
        return [s["plan"].outbuf, [c.nbytes for c in cs][:63]]
    rs = [pipeline.Retriever(c) for c in s["streams"]]
    rounds = [pipeline.retrieve_batch([(r, t[k]) for r, t in zip(rs, s["targets"])], pinned=True)
              for k in range(case["rounds"])]
    torch.cuda.current_stream().synchronize()  # errors() may be read then, and the batches' buffers given back
    if any(e for b in rounds for e in b.errors()):
        raise RuntimeError("malformed stream")
    return [b.outs for b in rounds]


# -------------------------------------------------------------------- work --
def _stream_bytes(n, item, eb, kind):
    """About how many bytes a field's stream takes: the bits that the codes of
    one value keep (the logarithm of its unpredictable part over the bound)
    and what the sparse planes above them cost."""
    sigma = {"mix": 1e-4, "density": 2e-4, "grf": 2e-3, "modes": 2e-4}[kind]
    bits = 0.6 + 1.15 * max(0.0, math.log2(sigma / eb) + 2.0)
    return n * min(bits, 8.0 * item) / 8.0


def work(case):
    """A compression reads the field and writes the stream; a decompression
    the reverse; a series of rounds reads the stream once in all and writes
    the field in each round, reading the one of the round before."""
    if case["kind"].startswith("batch"):
        parts = [_spec(case, i) for i in range(case["fields"])]
        fs = [(math.prod(shape), ITEM[dt], eb, kind) for shape, dt, kind, eb in parts]
    else:
        eb = case["eb"]
        fs = [(case["nx"] * case["ny"] * case["nz"], ITEM[case["dtype"]], eb, case["field"])]
    b = f = 0.0
    for n, item, eb, kind in fs:
        z = _stream_bytes(n, item, eb, kind)
        if case["kind"] in ("retrieve", "batch_retrieve"):
            b += z + (2 * case["rounds"] - 1) * n * item
            f += 12.0 * n * case["rounds"]
        else:
            b += z + n * item
            f += 16.0 * n
    return {"bytes": b, "flops": f}


def exact(case, seed):
    """The field itself, in 64 bits: what every decompression approximates
    (None for a first look coarser than 1e-2, which is none).  A stream is
    bytes and has no such value."""
    if case["kind"] in ("compress", "batch_compress"):
        return None
    fs, _ = _inputs(case, seed)
    fs = [f.double() for f in fs]
    if case["kind"] == "decompress":
        return fs[0]
    near = [case["first"] * 10.0 ** -k <= 1.5e-2 for k in range(case["rounds"])]
    if case["kind"] == "retrieve":
        return [fs[0] if ok else None for ok in near]
    return [[f if ok else None for f in fs] for ok in near]
