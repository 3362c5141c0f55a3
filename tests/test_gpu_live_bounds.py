"""Which planes are left out, at the codes where a power of two decides it, and
over the turns of a batch whose codes grow and shrink.  What is not written holds
ones, so that a byte too many left out shows.  Tolerance: none."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pl():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from prism_amd import pipeline
    return pipeline


def P(t, byte=0):
    return C.c_void_p(t.data_ptr() + byte)


def ones(n, dtype=torch.uint8):
    return torch.full((max(1, -(-int(n) // dtype.itemsize) * dtype.itemsize),), 255, dtype=torch.uint8,
                      device="cuda").view(dtype)


@pytest.mark.parametrize("mode", ["NB", "SM"])
@pytest.mark.parametrize("many", [False, True])
def test_codes_at_powers_of_two(pl, mode, many):
    """The largest codes of each level are -2^b, 2^b - 1 or both, by themselves or
    everywhere, with the magnitudes c ^ (c >> 31) that the predictor leaves."""
    from prism_amd import _lib
    lb, st = _lib.lib(), pl._stream()
    mode = {"NB": _lib.PA_MODE_NB, "SM": _lib.PA_MODE_SM}[mode]
    L = pl.layout(130, 97, 141)
    starts = [L.prefix[lv] for lv in range(4)]
    counts = [L.n - L.cnt[0], L.cnt[0] - L.cnt[1], L.cnt[1] - L.cnt[2], L.cnt[2] - L.n4]
    nws = lb.pa_encode_workspace(C.byref(L))

    def encode(qc, words):
        bp, out, cum, size, ws = ones(L.host_size), ones(lb.pa_compress_bound(C.byref(L), 8)), ones(1024), ones(16), ones(nws)
        a = (C.byref(L), P(out), P(cum), P(size), P(ws), nws, st)
        if words is None:
            _lib.check(lb.pa_bitshuffle(P(qc), C.byref(L), mode, P(bp), st))
            _lib.check(lb.pa_lossless_encode(P(bp), *a))
        else:
            _lib.check(lb.pa_encode_prepare(C.byref(L), P(ws), nws, st))
            ws.view(torch.int64)[1 + L.nchunks + 16 * 3] = words
            _lib.check(lb.pa_bitshuffle_live(P(qc), C.byref(L), mode, P(bp), P(ws), nws, st))
            _lib.check(lb.pa_lossless_encode_live(P(bp), *a))
        n = int(size.view(torch.int64)[0])
        return out[:n].clone(), cum

    g = torch.Generator(device="cuda").manual_seed(5)
    for b in range(32):
        for which in ((-2 ** b,), (2 ** b - 1,), (-2 ** b, 2 ** b - 1)):
            qc = torch.zeros(L.code_len, dtype=torch.int32, device="cuda")
            mags = [0, 0]
            for lv in range(4):
                bl = b if lv == 0 else (b + 5 * lv) % 32  # (each level another power)
                vals = [-2 ** bl if v < 0 else 2 ** bl - 1 for v in which]
                seg = qc[starts[lv]:starts[lv] + counts[lv]]
                if many:
                    at = torch.randint(0, 3 * len(vals), (counts[lv],), device="cuda", generator=g)
                    for i, v in enumerate(vals):
                        seg[at == i] = v
                else:
                    for i, v in enumerate(vals):
                        seg[(counts[lv] * (2 * i + 1)) // 4] = v
                for v in vals:
                    mags[min(lv, 1)] |= v ^ (v >> 31)
            words = mags[0] | (mags[1] << 32)
            want, got = encode(qc, None), encode(qc, words)
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (b, which)


def test_turns_of_a_batch(pl, monkeypatch):
    """The planes that a batch leaves out follow its codes from turn to turn, up and
    down, by graph and again with new fields and bounds."""
    shapes = [(304, 304, 304), (304, 304, 288), (70, 80), (33, 40, 65)]
    types = [torch.float32, torch.float64] * 2
    g = torch.Generator(device="cuda").manual_seed(7)

    def fields(spike):
        out = []
        for s, t in zip(shapes, types):
            d = torch.zeros(s, dtype=t, device="cuda")
            for axis, n in enumerate(s):
                d += torch.sin(torch.linspace(0, 4 + axis, n, dtype=t, device="cuda")).view(
                    [-1 if i == axis else 1 for i in range(len(s))])
            d += 0.01 * torch.rand(s, dtype=t, device="cuda", generator=g)
            d.view(-1)[d.numel() // 3] += spike
            out.append(d)
        return out

    turns = [(fields(0.0), 1e-1), (fields(0.0), 1e-6), (fields(0.0), 1e-2), (fields(40.0), 1e-5), (fields(0.0), 1e-1)]
    want = [[pl.compress(d, e).stream.cpu() for d in ds] for ds, e in turns]
    with monkeypatch.context() as m:
        m.setattr(pl, "_empty", ones)  # the plan's workspace, planes and magnitudes among it
        b = pl.BatchCompressor(turns[0][0], [turns[0][1]] * 4, graph=True)
    for k, (ds, e) in enumerate(turns):
        for again in range(2):
            res = b.run(ds, [e] * 4) if again == 0 else b.run()
            for i, (r, w) in enumerate(zip(res, want[k])):
                assert torch.equal(r.stream.cpu(), w), (k, again, i)
