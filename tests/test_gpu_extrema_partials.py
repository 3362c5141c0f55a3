"""Extremes planted where the extrema workgroups beside the tuner, which leave
partial results, can lose them: 3-D fields with tuner samples (1-D and 2-D ones
take pa_extrema), with fewer partial results than the finishing workgroup has
lanes, with several for each lane, and with as many as there can be, each then
over more than one batch of loads.  Tolerance: none."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BATCH, MOST, LANES = 2048, 2048, 256  # vectors of a batch of loads; partial results at most; finishing lanes


def spans(n, item):
    """(vectors of 16 bytes, vectors of a workgroup, workgroups), as they are cut."""
    nv = n * item // 16
    span = max(-(-nv // MOST), BATCH)
    return nv, span, -(-nv // span)


@pytest.mark.parametrize("shape,dtype,few", [((65, 67, 101), torch.float32, True), ((161, 163, 203), torch.float32, False),
                                             ((161, 163, 203), torch.float64, False),
                                             ((257, 259, 261), torch.float32, False),
                                             ((257, 259, 261), torch.float64, False)])
def test_planted_extremes(shape, dtype, few):
    from prism_amd import _lib, pipeline as pl
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nz, ny, nx = shape
    n, item = nx * ny * nz, dtype.itemsize
    V = 16 // item
    nv, span, groups = spans(n, item)
    assert n % V != 0 and (groups < LANES if few else groups > LANES), (n, groups)
    assert groups <= MOST and (span > BATCH) == (shape[0] == 257)
    print("CASE planted extremes", shape, dtype, groups, span, flush=True)
    # values at the ends of the field and of its vectors, at the ends of spans that the
    # first, second and last trips of the finishing lanes take, and inside a span
    vectors = [0, BATCH, nv - 1]
    for k in {1, min(LANES - 1, groups - 1), min(LANES, groups - 1), min(2 * LANES + 3, groups - 1), groups // 2, groups - 1}:
        vectors += [k * span - 1, k * span, k * span + min(span, nv - k * span) // 2]
    places = sorted({v * V + e for v in vectors for e in (0, V - 1)} | {nv * V, n - 1})
    g = torch.Generator(device="cuda").manual_seed(11)
    d = torch.rand(n, dtype=dtype, device="cuda", generator=g)
    L = pl.layout(nx, ny, nz)
    lb = _lib.lib()
    full = lb.pa_autotune_workspace(C.byref(L))
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    out = torch.empty(32, dtype=torch.float64, device="cuda")
    p = lambda t, byte=0: C.c_void_p(t.data_ptr() + byte)
    got, want = [], []
    for i, at in enumerate(places):
        other = places[(7 * i + 3) % len(places)]
        if other == at:
            other = places[i - 1]
        keep = d[at].clone(), d[other].clone()
        d[at], d[other] = -2.0 - i, 3.0 + i
        for nbytes in (full, full - 8):  # partial results; the two keys
            out.fill_(-1.0)
            _lib.check(lb.pa_extrema_autotune(p(d), pl.DTYPES[dtype], C.byref(L), p(out), 1e-3, p(out, 64), None,
                                              p(out, 48), p(ws), nbytes, pl._stream()))
            got.append(out[[0, 1, 9]].clone())  # min, max, and the range of the bounds
            want.append((-2.0 - i, 3.0 + i, 5.0 + 2 * i))
        d[at], d[other] = keep
    assert torch.equal(torch.stack(got).cpu(), torch.tensor(want, dtype=torch.float64))
