"""What the host-side calls wait for, seen from a stream that is still busy
when they are made."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pl():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from prism_amd import pipeline
    return pipeline


def fields(pl, rel):
    d = torch.sin(torch.linspace(0, 40, 17 * 33 * 65, dtype=torch.float64, device="cuda")).view(17, 33, 65)
    c = pl.compress(d, 1e-3, rel=rel, progressive=False)
    return c, pl.decompress(c)  # (a first call: everything is loaded)


def busy(stream):
    """At least 10 ms of work ahead of what the stream gets next (a host call takes
    well below a millisecond); the event fires when it is done."""
    torch.cuda._sleep(20_000_000)
    e = torch.cuda.Event()
    e.record()
    assert not stream.query(), "the stream should be busy"
    return e


class Failing:
    """The library with one call that fails."""

    def __init__(self, lib, name, status):
        self.lib, self.name, self.status = lib, name, status

    def __getattr__(self, name):
        return (lambda *a: self.status) if name == self.name else getattr(self.lib, name)


@pytest.mark.parametrize("name", ["pa_lossless_decode", "pa_inverse_bitshuffle"])
def test_a_failing_decompression_leaves_no_copy_behind(pl, monkeypatch, name):
    """The copy of the range to the thread's buffer has arrived when the call
    raises, so that the thread's next read, on any stream, has the buffer alone."""
    from prism_amd import _lib
    c, want = fields(pl, True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    failing = Failing(pl.lib(), name, _lib.PA_ERR_WORKSPACE)
    with torch.cuda.stream(s), monkeypatch.context() as m:
        m.setattr(pl, "lib", lambda: failing)
        busy(s)
        with pytest.raises(_lib.PrismError):
            pl.decompress(c)
        if name == "pa_lossless_decode":  # nothing was queued behind the copy
            assert s.query()
    # ... and a value written after the call stays
    pl._TLS.pinned[:8] = 7
    s.synchronize()
    assert pl._TLS.pinned[:8].tolist() == [7] * 8
    assert torch.equal(pl.decompress(c), want)


def test_absolute_bounds_wait_for_nothing(pl):
    c, want = fields(pl, False)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        before = busy(s)
        out = pl.decompress(c, check_stream=False)
        assert not before.query()
    s.synchronize()
    assert torch.equal(out, want)
