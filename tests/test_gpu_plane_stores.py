"""Rounds of 2-D fields below and above the size from which their delta form
writes past the caches, alone and by the sum of a batch.  Tolerance: none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pl():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from prism_amd import pipeline
    return pipeline


def field(ny, nx, dtype):
    y, x = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    return (np.sin(0.01 * x) * np.cos(0.02 * y) + 1e-3 * np.random.default_rng(nx).random((ny, nx))).astype(dtype)[None]


# 100 MiB are 13107200 float64 and 26214400 float32 values
@pytest.mark.parametrize("dtype,shape", [(np.float64, (3600, 3640)), (np.float64, (3600, 3641)), (np.float32, (5120, 5121)),
                                         (np.float32, (17, 1003)), (np.float64, (130, 64))])
def test_rounds_of_planes(pl, oracle, dtype, shape):
    print("CASE plane rounds", shape, dtype.__name__, flush=True)
    data, rel = field(*shape, dtype), 1e-4
    s_o, _ = oracle.compress(data, rel, mode=0)
    c = pl.compress(torch.from_numpy(data).cuda(), rel)
    assert np.array_equal(c.stream.cpu().numpy(), s_o)
    po, rv = oracle.Progressive(s_o, data.shape, dtype, rel, corrected=True), pl.Retriever(c)
    for t in (1e-2, rel):
        assert np.array_equal(rv.retrieve(t).cpu().numpy().view(np.uint8), po.retrieve(t)[0].view(np.uint8)), t


def test_batches_of_planes(pl):
    data = [field(2000, 2100, np.float64), field(2100, 2000, np.float32), field(900, 1000, np.float64),
            field(2500, 2050, np.float64)]
    cs = [pl.compress(torch.from_numpy(d).cuda(), 1e-4) for d in data]
    for n in (3, 4):  # 55 MB, then 126 (one field is there twice)
        many = cs[:n] + (cs[:1] if n == 4 else [])
        batch, alone = [pl.Retriever(c) for c in many], [pl.Retriever(c) for c in many]
        for t in (1e-2, 1e-4):
            for got, r in zip(pl.retrieve_batch([(r, t) for r in batch]).outs, alone):
                assert torch.equal(got, r.retrieve(t)), (n, t)
