"""Compression that neither writes nor reads the bit-planes which hold no bit:
the stream must equal, byte for byte, the one from whole planes, which the
parity tests pin to the oracle.  Tolerance: none."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pl():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from prism_amd import pipeline
    return pipeline


def field(shape, dtype, spike):
    g = torch.Generator(device="cuda").manual_seed(17)
    d = 0.01 * torch.rand(shape, dtype=dtype, device="cuda", generator=g)
    for axis, n in enumerate(shape):
        d += torch.sin(torch.linspace(0, 5 + axis, n, dtype=dtype, device="cuda")).view(
            [-1 if i == axis else 1 for i in range(len(shape))])
    if spike:  # codes that one workgroup alone finds large
        d.view(-1)[d.numel() * 2 // 3] += spike
    return d


# planes of less than a chunk, of some chunks and of many; 2-D and 1-D fields,
# which leave no magnitudes
@pytest.mark.parametrize("shape", [(33, 17, 18), (64, 64, 64), (130, 97, 141), (160, 176, 192), (300, 400), (300000,)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("progressive", [True, False])
def test_live_planes_equal_whole_planes(pl, monkeypatch, shape, dtype, progressive):
    print("CASE live planes", shape, dtype, progressive, flush=True)
    # bounds that leave many, some and few planes zero; a spike in one tile
    for eb, spike in ((1e-1, 0.0), (1e-3, 0.0), (1e-3, 50.0), (1e-6, 0.0)):
        d = field(shape, dtype, spike)
        want = pl.compress(d, eb, progressive=progressive).stream.cpu()
        with monkeypatch.context() as m:
            m.setattr(pl.lib(), "pa_live_planes", lambda L: 1)
            # what stays unwritten holds ones
            m.setattr(pl, "_empty", lambda n, dtype=torch.uint8: torch.full((n,), 255, dtype=dtype, device="cuda"))
            got = pl.compress(d, eb, progressive=progressive).stream.cpu()
        assert torch.equal(got, want), (eb, spike)


def test_live_planes_of_a_batch(pl):
    """A batch past the size from which planes are left out, with fields of
    every dimension, by graph and again; each field alone is below it."""
    shapes = [(304, 304, 304), (304, 304, 288), (300, 400), (40, 33, 65), (5000,)]
    data = [field(s, t, 0.0) for s, t in zip(shapes, [torch.float32, torch.float64] * 3)]
    ebs = [1e-3, 1e-5, 1e-3, 1e-2, 1e-4]
    want = [pl.compress(t, e).stream.cpu() for t, e in zip(data, ebs)]
    b = pl.BatchCompressor(data, ebs, graph=True)
    for turn in range(2):
        torch.full((1 << 20,), 255, dtype=torch.uint8, device="cuda")  # eager work between replays
        for i, (g, w) in enumerate(zip(b.run(), want)):
            assert torch.equal(g.stream.cpu(), w), (turn, i)
        data = [t * 2 + 1 for t in data]
        want = [pl.compress(t, e).stream.cpu() for t, e in zip(data, ebs)]
        for i, (g, w) in enumerate(zip(b.run(data, ebs), want)):
            assert torch.equal(g.stream.cpu(), w), (turn, "rebound", i)
