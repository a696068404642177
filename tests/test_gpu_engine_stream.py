"""The engine stream context: torch's current stream and device as
``torch.cuda.stream`` leaves them, also nested, after an exception and as a
decorator; ``stream_handle`` is the current stream's handle."""
import pytest

pytestmark = pytest.mark.gpu


def test_engine_stream_switches_and_restores():
    import torch

    from pih_amd.device import engine_stream, stream, stream_handle

    before = torch.cuda.current_stream()
    with pytest.raises(RuntimeError, match="explicit stream"):
        stream_handle()
    other = torch.cuda.Stream()
    with engine_stream() as s:
        assert s is stream() and torch.cuda.current_stream() == s and stream_handle() == s.cuda_stream
        with torch.cuda.stream(other):
            assert stream_handle() == other.cuda_stream
            with engine_stream():
                assert torch.cuda.current_stream() == s
            assert torch.cuda.current_stream() == other
        assert torch.cuda.current_stream() == s
    assert torch.cuda.current_stream() == before
    with pytest.raises(KeyError):
        with engine_stream():
            raise KeyError
    assert torch.cuda.current_stream() == before

    @engine_stream()
    def depth(n):
        assert torch.cuda.current_stream() == stream()
        return depth(n - 1) if n else 0

    assert depth(2) == 0 and torch.cuda.current_stream() == before


def test_engine_stream_context_is_entered_once():
    """A second entry, from inside, afterwards or from another thread, is
    refused and leaves every thread on the stream it had."""
    import threading

    import torch

    from pih_amd.device import engine_stream, stream

    before = torch.cuda.current_stream()
    ctx, seen = engine_stream(), []

    def other_thread():
        try:
            ctx.__enter__()
        except RuntimeError as e:
            seen.append((str(e), torch.cuda.current_stream() == before))

    with ctx:
        with pytest.raises(RuntimeError, match="entered once"):
            ctx.__enter__()
        t = threading.Thread(target=other_thread)
        t.start()
        t.join()
        assert torch.cuda.current_stream() == stream()
    assert torch.cuda.current_stream() == before and len(seen) == 1 and seen[0][1]
    with pytest.raises(RuntimeError, match="entered once"):
        with ctx:
            pass
    assert torch.cuda.current_stream() == before
