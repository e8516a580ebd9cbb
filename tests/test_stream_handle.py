"""The current stream's handle with and without torch's raw accessors (no GPU needed: the
accessors are stand-ins)."""
import pytest

torch = pytest.importorskip("torch")

from asteriy_2d_amd import native  # noqa: E402


class _Stream:
    cuda_stream = 1234


@pytest.mark.parametrize("missing", [(), ("_cuda_getCurrentRawStream",), ("_cuda_getDevice",),
                                     ("_cuda_getCurrentRawStream", "_cuda_getDevice")])
@pytest.mark.parametrize("initialized", [True, False])
def test_current_stream(monkeypatch, missing, initialized):
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: initialized)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: _Stream())
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 3, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: 1000 + d, raising=False)
    for name in missing:
        monkeypatch.delattr(torch._C, name)
    assert native.stream_handle() == (1003 if initialized and not missing else 1234)
    assert native.stream_handle(_Stream()) == 1234
