"""A torch without the internals that the shortcuts ask: the general paths."""
import pytest
import torch

from temgymcore_amd import _lib, gaussian


@pytest.mark.parametrize("name", ["_len_torch_dispatch_stack", "_len_torch_function_stack", "_get_tracing_state"])
def test_pack_takes_the_torch_operations(monkeypatch, name):
    assert gaussian._no_transform()
    monkeypatch.delattr(torch._C, name)
    assert not gaussian._no_transform()


def test_lookups_by_the_public_functions(monkeypatch):
    class Stream:
        cuda_stream = 77

    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream)
    monkeypatch.setattr(_lib, "_get_device", None)
    monkeypatch.setattr(_lib, "_get_raw_stream", None)
    assert _lib.stream_ptr(torch.device("cuda", 3)) == 77
    assert _lib.require_device() == torch.device("cuda", 3)
