"""Argument handling of the Python wrappers: the verdicts on tensors, and the stream a call uses."""
import pytest
import torch

from dadgpt_amd import attention as A


def test_ptrs_verdicts_without_a_device():
    """A tensor that fails any check gets _require's own error; None passes as None."""
    good = torch.zeros(8)
    assert A._ptrs(torch.float32, 8, (None,), ("x",)) == [None]
    for bad, error, text in ((good, ValueError, "x must be a device tensor"),
                             ([1.0], TypeError, "x must be a torch.Tensor"),
                             (torch.nn.Parameter(good), ValueError, "device tensor")):
        with pytest.raises(error, match=text):
            A._ptrs(torch.float32, 8, (None, bad), ("y", "x"))


@pytest.mark.gpu
def test_ptrs_verdicts_on_the_device(gpu):
    t = torch.zeros(4, 8, device="cuda")
    p = torch.nn.Parameter(t)
    assert A._ptrs(torch.float32, 32, (t, None, p), "abc") == [t.data_ptr(), None, p.data_ptr()]
    for bad, error, text in ((t.half(), TypeError, "b must be torch.float32"),
                             (t.t(), ValueError, "b must be contiguous"),
                             (t[:3], ValueError, "b has 24 elements, needs 32")):
        with pytest.raises(error, match=text):
            A._ptrs(torch.float32, 32, (t, bad), "ab")


@pytest.mark.gpu
def test_calls_follow_the_current_stream(gpu):
    """None is torch's current stream (the default one is the null stream), also inside a stream
    context; a Stream object is used as given."""
    assert A._stream_ptr(None) is None
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert A._stream_ptr(None) == s.cuda_stream
    assert A._stream_ptr(s) == s.cuda_stream
    assert A._stream_ptr(None) == (torch.cuda.current_stream().cuda_stream or None)
