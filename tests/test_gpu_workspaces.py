"""Workspaces at the sizes that the header gives: accepted from there on, not
written past, and refused below.  Tolerance: none."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pa():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from prism_amd import _lib, pipeline
    return _lib, pipeline


def P(t, byte=0):
    return C.c_void_p(t.data_ptr() + byte)


def sample_blocks(*axes):
    n = 1
    for d in axes:
        n *= (d // 2 - 8) // 128 + (d - 9 - d // 2) // 128 + 1
    return n


# 1, 27 and 9 sample blocks; fewer values than one workgroup's loads, and more
# extrema workgroups than the finishing one has lanes
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(17, 18, 19), (273, 290, 273), (160, 300, 520)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_extrema_beside_a_tuner_workspace(pa, shape, dtype):
    """The tuner's sums, one double per sample block and candidate, are workspace
    enough: the extrema then meet behind the result."""
    _lib, pl = pa
    print("CASE tuner workspace", shape, dtype, flush=True)
    nz, ny, nx = shape
    L = pl.layout(nx, ny, nz)
    need = 8 * 15 * sample_blocks(nx, ny, nz)
    g = torch.Generator(device="cuda").manual_seed(3)
    d = torch.rand(shape, dtype=dtype, device="cuda", generator=g)
    d.view(-1)[-1], d.view(-1)[d.numel() // 3] = -3.0, 5.0

    def call(ws_bytes):
        # result, scores, flags and bounds; the workspace's bytes past its size are watched
        r = torch.full((4 + 15 + 1 + 16,), -1.0, dtype=torch.float64, device="cuda")
        ws = torch.full((max(ws_bytes, need) + 256,), 255, dtype=torch.uint8, device="cuda")
        _lib.check(_lib.lib().pa_extrema_autotune(P(d), pl.DTYPES[dtype], C.byref(L), P(r), 1e-3, P(r, 160), P(r, 32),
                                                  P(r, 152), P(ws), ws_bytes, pl._stream()))
        torch.cuda.synchronize()
        assert bool((ws[ws_bytes:] == 255).all())
        r[2:4] = 0.0  # scratch
        return r

    want = call(_lib.lib().pa_autotune_workspace(C.byref(L)))
    assert want[0:2].tolist() == [-3.0, 5.0]
    for ws_bytes in (need, need + 8 * 100):
        assert torch.equal(call(ws_bytes).view(torch.int64), want.view(torch.int64)), ws_bytes


def test_short_tuner_workspaces_are_refused():
    from prism_amd import _lib, pipeline as pl
    L = pl.layout(273, 290, 273)
    host = (C.c_double * 64)()  # never reached
    p = C.c_void_p((C.addressof(host) + 15) // 16 * 16)
    need = 8 * 15 * sample_blocks(273, 290, 273)
    assert need <= _lib.lib().pa_autotune_workspace(C.byref(L))
    for ws, nbytes in ((p, need - 1), (p, 0), (None, need)):
        assert _lib.lib().pa_extrema_autotune(p, 8, C.byref(L), p, 1e-3, p, p, p, ws, nbytes, None) == _lib.PA_ERR_WORKSPACE
        assert _lib.lib().pa_autotune(p, 8, C.byref(L), p, p, ws, nbytes, None) == _lib.PA_ERR_WORKSPACE


def test_short_encoder_workspaces_are_refused():
    """By every call of the compression that leaves zero planes out; the plain
    encoder needs the words before the code magnitudes alone."""
    from prism_amd import _lib, pipeline as pl
    lb = _lib.lib()
    for L in (pl.layout(130, 97, 141), pl.layout(300, 400, 1)):
        host = (C.c_double * 64)()  # never reached
        p = C.c_void_p((C.addressof(host) + 15) // 16 * 16)
        need, plain = lb.pa_encode_workspace(C.byref(L)), 8 * (1 + L.nchunks)
        assert need > plain
        for ws, nbytes in ((p, need - 1), (p, plain), (p, 0), (None, need), (C.c_void_p(p.value + 4), need)):
            calls = (lb.pa_encode_prepare(C.byref(L), ws, nbytes, None),
                     lb.pa_spline_construct_live(p, 8, C.byref(L), p, p, p, p, ws, nbytes, None),
                     lb.pa_bitshuffle_live(p, C.byref(L), 0, p, ws, nbytes, None),
                     lb.pa_lossless_encode_live(p, C.byref(L), p, p, p, ws, nbytes, None))
            assert calls == (_lib.PA_ERR_WORKSPACE,) * 4, (nbytes, calls)
        assert lb.pa_lossless_encode(p, C.byref(L), p, p, p, p, plain - 1, None) == _lib.PA_ERR_WORKSPACE
