"""The Python module on a torch built without GPU support: it imports, and the host-only functions work."""
import importlib.util
import types

import pytest
import torch

import gfr_moe


@pytest.fixture
def without_gpu_build(monkeypatch):
    """The module loaded afresh with torch._C's GPU-only names absent."""
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    spec = importlib.util.spec_from_file_location("gfr_moe_without_gpu", gfr_moe.__file__)
    m = importlib.util.module_from_spec(spec)
    monkeypatch.setitem(__import__("sys").modules, spec.name, m)
    spec.loader.exec_module(m)
    return m


def test_host_functions_without_a_gpu_build(without_gpu_build):
    i32, f16 = torch.int32, torch.float16
    w = without_gpu_build.Exl3Experts(
        gt=torch.zeros((1, 16, 16, 32), dtype=i32), ut=torch.zeros((1, 16, 16, 32), dtype=i32),
        dt=torch.zeros((1, 16, 16, 32), dtype=i32), suh_g=torch.zeros((1, 256), dtype=f16),
        suh_u=torch.zeros((1, 256), dtype=f16), suh_d=torch.zeros((1, 256), dtype=f16),
        svh_g=torch.zeros((1, 256), dtype=f16), svh_u=torch.zeros((1, 256), dtype=f16),
        svh_d=torch.zeros((1, 256), dtype=f16), bits=4)
    assert (w.experts, w.hidden, w.inter) == (1, 256, 256)
    with pytest.raises(ValueError, match="on GPU"):
        w.check()
    assert b"gfx950" in without_gpu_build.lib().gfr_version()


def test_stream_handles_without_the_raw_call(without_gpu_build, monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    assert without_gpu_build._stream() == 77
    assert without_gpu_build._stream(types.SimpleNamespace(cuda_stream=5)) == 5
