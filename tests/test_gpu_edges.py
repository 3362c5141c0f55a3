"""Edges of the tile groups, the extrema partials and the encoder's write,
against the oracle.  Tolerance: none."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pa():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from prism_amd import _lib, pipeline
    return _lib, pipeline


def P(t):
    return C.c_void_p(t.data_ptr())


# x extents around one, two and three tiles (float32 reconstruction takes
# tiles in pairs, the last one alone where their number is odd) and rows of whole
# 128-byte lines and not; y and z with full and cut tiles
@pytest.mark.parametrize("nx", [15, 16, 17, 31, 32, 33, 48, 49, 64, 80])
@pytest.mark.parametrize("nz,ny", [(16, 32), (33, 17), (7, 18)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_tile_groups(pa, oracle, nz, ny, nx, dtype):
    _, pipe = pa
    print("CASE tile groups", nz, ny, nx, dtype.__name__, flush=True)
    z, y, x = np.meshgrid(*(np.arange(n) for n in (nz, ny, nx)), indexing="ij")
    data = (np.sin(0.3 * x + 0.1 * z) * np.cos(0.2 * y) + 1e-3 * np.random.default_rng(nx).random((nz, ny, nx))).astype(dtype)
    rel = 1e-4
    s_o, _ = oracle.compress(data, rel, mode=0)
    c = pipe.compress(torch.from_numpy(data).cuda(), rel)
    assert np.array_equal(c.stream.cpu().numpy(), s_o)
    po, rv = oracle.Progressive(s_o, data.shape, dtype, rel, corrected=True), pipe.Retriever(c)
    for t in (1e-1, 1e-3, rel):  # codes from the planes, in 16 and in 32 bits
        assert np.array_equal(rv.retrieve(t).cpu().numpy().view(np.uint8), po.retrieve(t)[0].view(np.uint8)), t
    s_o, _ = oracle.compress(data, rel, mode=1)
    c = pipe.compress(torch.from_numpy(data).cuda(), rel, progressive=False)
    assert np.array_equal(pipe.decompress(c).cpu().numpy().view(np.uint8),
                          oracle.decompress(s_o, data.shape, dtype, rel).view(np.uint8))


# fewer values than a workgroup's first loads, its multiples, and more
# workgroups than there are partial results
@pytest.mark.parametrize("n", [2, 1023, 4096, 4097, 65537, (1 << 21) + 3, (1 << 25) + 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_extrema_ends(pa, n, dtype):
    _, pipe = pa
    print("CASE extrema", n, dtype, flush=True)
    for lo, hi in ((0, n - 1), (n - 1, 0), (n // 2, n // 2 - 1)):
        d = torch.linspace(-1, 1, n, dtype=dtype, device="cuda")
        d[lo], d[hi] = -3.0, 5.0
        assert pipe.extrema(d).tolist()[:2] == [-3.0, 5.0]
        assert pipe.compress(d, 1e-2).range == 8.0


# shares of non-zero bytes from which chunks are zero-eliminated with full
# steps and a long tail up to those that are stored raw; planes whose last
# chunk ends at any byte of a 16-byte unit
@pytest.mark.parametrize("share", [0.003, 0.3, 0.8, 0.97, 0.999, 1.0])
@pytest.mark.parametrize("shape", [(1, 1, 17), (1, 1, 1003), (23, 29, 31), (70, 66, 129)])
def test_encoder_writes(pa, oracle, share, shape):
    _lib, _ = pa
    print("CASE encoder", share, shape, flush=True)
    nz, ny, nx = shape
    L, Lo = _lib.layout(nx, ny, nz), oracle.layout(nx, ny, nz)
    rng = np.random.default_rng(int(1000 * share) + nx)
    n = L.host_size
    bp = np.where(rng.random(n) < share, rng.integers(1, 256, n), 0).astype(np.uint8)
    bp[(n // 2) // 16384 * 16384:][:16384] = 0
    want, cum = oracle.lossless_encode(bp, Lo)
    for poison in (0, 255):  # bytes around the stream stay as they are
        out = torch.full((_lib.lib().pa_compress_bound(C.byref(L), 8) + 64,), poison, dtype=torch.uint8, device="cuda")
        cumd = torch.zeros(128, dtype=torch.int64, device="cuda")
        sz = torch.zeros(2, dtype=torch.int64, device="cuda")
        ws = torch.empty(_lib.lib().pa_encode_workspace(C.byref(L)), dtype=torch.uint8, device="cuda")
        bpd = torch.from_numpy(bp).cuda()
        _lib.check(_lib.lib().pa_lossless_encode(P(bpd), C.byref(L), P(out), P(cumd), P(sz), P(ws), ws.numel(),
                                                 C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        m = int(sz[0])
        got = out.cpu().numpy()
        assert m + (-m) % 8 == want.size and np.array_equal(got[:m], want[:m])
        assert (got[m:] == poison).all()
        assert np.array_equal(cumd.cpu().numpy().view(np.uint64), cum)
