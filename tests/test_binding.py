"""The Python binding's own parts that need no GPU."""
import types

import pytest


def test_stream_of_a_torch_with_and_without_the_raw_getters(pkg):
    public = types.SimpleNamespace(current_stream=lambda: types.SimpleNamespace(cuda_stream=7))
    raw = types.SimpleNamespace(_cuda_getDevice=lambda: 3, _cuda_getCurrentRawStream=lambda device: 100 + device)
    assert pkg._stream_getter(types.SimpleNamespace(_C=raw, cuda=public))() == 103
    for missing in ("_cuda_getDevice", "_cuda_getCurrentRawStream"):
        some = types.SimpleNamespace(**{k: v for k, v in vars(raw).items() if k != missing})
        assert pkg._stream_getter(types.SimpleNamespace(_C=some, cuda=public))() == 7


def test_a_missing_weight_is_the_librarys_error(pkg, monkeypatch):
    torch = pytest.importorskip("torch")
    monkeypatch.setattr(pkg, "_raw_stream", lambda: 0)
    ws = torch.empty(int(pkg.lib().w4a32_workspace_bytes_n(1, 64, 32)) + 256, dtype=torch.uint8)
    with pytest.raises(pkg.W4A32Error, match="w4a32_matmul_ws"):  # refused before anything is launched
        pkg.matmul_ws(torch.zeros((1, 64)), None, 32, ws=ws, out=torch.zeros((1, 32)))


@pytest.mark.gpu
def test_stream_is_the_current_one(pkg):
    import torch

    assert pkg._stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert pkg._stream() == side.cuda_stream
    assert pkg._stream() == torch.cuda.current_stream().cuda_stream != side.cuda_stream
