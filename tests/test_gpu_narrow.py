"""Reconstruction of fields of one tile along x, whose float32 workgroups take
one tile: even and odd numbers of tiles, rows of one to sixteen
values, alone and beside wider fields.  Against the oracle, tolerance: none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))


def field(nz, ny, nx, dtype):
    z, y, x = np.meshgrid(*(np.arange(n) for n in (nz, ny, nx)), indexing="ij")
    noise = np.random.default_rng(nx + 100 * ny + 10000 * nz).random((nz, ny, nx))
    return (np.sin(0.3 * x + 0.1 * z) * np.cos(0.2 * y) + 1e-2 * noise).astype(dtype)


# 1, 2, 3, 6, 9 and 35 tiles
@pytest.mark.parametrize("nz,ny", [(16, 9), (2, 17), (40, 16), (17, 33), (40, 47), (70, 112)])
@pytest.mark.parametrize("nx", [1, 3, 15, 16])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_one_tile_along_x(oracle, nz, ny, nx, dtype):
    from prism_amd import pipeline as pl
    print("CASE narrow", nz, ny, nx, dtype.__name__, flush=True)
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    data, rel = field(nz, ny, nx, dtype), 1e-5
    s_o, _ = oracle.compress(data, rel, mode=1)
    c = pl.compress(torch.from_numpy(data).cuda(), rel, progressive=False)
    assert np.array_equal(c.stream.cpu().numpy(), s_o)
    assert same(pl.decompress(c).cpu().numpy(), oracle.decompress(s_o, data.shape, dtype, rel))
    s_o, _ = oracle.compress(data, rel, mode=0)
    c = pl.compress(torch.from_numpy(data).cuda(), rel)
    # in one launch with a wider field and one of the other type
    others = [pl.compress(torch.from_numpy(field(18, 20, n, t)).cuda(), rel)
              for n, t in ((49, dtype), (16, np.float32), (16, np.float64))]
    batch = [pl.Retriever(x) for x in [others[0], c] + others[1:]]
    alone = [pl.Retriever(x) for x in others]
    po, rv = oracle.Progressive(s_o, data.shape, dtype, rel, corrected=True), pl.Retriever(c)
    for t in (1e-1, 3e-2, 1e-4, rel):  # codes in 32 bits, from the planes, in 16 bits
        want = po.retrieve(t)[0]
        assert same(rv.retrieve(t).cpu().numpy(), want), t
        outs = pl.retrieve_batch([(r, t) for r in batch]).outs
        assert same(outs[1].cpu().numpy(), want), t
        for got, r in zip([outs[0]] + outs[2:], alone):
            assert torch.equal(got, r.retrieve(t)), t
