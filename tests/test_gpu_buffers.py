"""The buffers of a retrieval: those of a large field are memory of their own,
those of a small one share a block of bounded size."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(5,), (17, 33, 65), (199, 200, 201), (200, 200, 210), (9000000,)])
def test_kept_buffers_hold_no_large_others(shape):
    from prism_amd import pipeline as pl
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    print("CASE buffers", shape, flush=True)
    d = torch.sin(torch.arange(torch.Size(shape).numel(), dtype=torch.float32, device="cuda")).view(shape)
    c = pl.compress(d, 1e-3)
    r = pl.Retriever(c)
    want = {"bp": r.L.host_size, "qc": 4 * r.L.code_len, "dws": pl.lib().pa_decode_workspace(pl.C.byref(r.L))}
    small = sum(want.values()) <= pl._ONE_BLOCK - 2048  # (512-byte starts)
    out = r.retrieve(1e-3)
    assert torch.equal(out.view(torch.int32), pl.decompress(c).view(torch.int32))  # all planes, in one round
    for name, nbytes in want.items():
        t = getattr(r, name)
        assert t.numel() * t.element_size() == nbytes, name
        assert getattr(r, name).data_ptr() == t.data_ptr() and t.data_ptr() % 512 == 0
        held = t.untyped_storage().nbytes()
        assert held <= pl._ONE_BLOCK if small else held == nbytes, (name, held)
