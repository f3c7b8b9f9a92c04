"""Calls with tensors in host memory end in an error on the host, whatever the runtime says about device -1 -- no GPU."""
import pytest
import torch


@pytest.fixture
def any_device_has_a_stream(monkeypatch):
    """The runtime of a machine with a GPU: the raw stream of device -1 is the current device's."""
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 0)


def test_mixer_calls_refuse_host_tensors(any_device_has_a_stream, monkeypatch):
    from exllamav3_amd import _lib, mix_ops
    reached = []
    lib = type("Lib", (), {"__getattr__": lambda self, name: lambda *a: reached.append(name) or 0})()
    monkeypatch.setattr(_lib, "mixlib", lambda: lib)
    f = torch.zeros
    i32 = lambda n: f(n, dtype=torch.int32)
    calls = [lambda: mix_ops.rms_norm_rows(f(4, 8), f(4, 8), None, f(8), 1e-5),
             lambda: mix_ops.embed(f(4, 8), f(4, 8), f(10, 8), i32(4), 1.0, f(8), 1e-5),
             lambda: mix_ops.polynorm(f(4, 8), f(4, 8), f(4), 1e-5),
             lambda: mix_ops.gla_out(f(4, 16), f(4, 2, 8), f(8), f(4, 16), 1e-5),
             lambda: mix_ops.gla_scan(f(4, 1, 8), f(1, 1, 64, 8), f(4, 64), f(4, 64), f(4, 8), f(4, 4), f(64, 4), None, i32(2), i32(1), i32(1), 1.0, 1.0, segments=(1, 16))]
    for call in calls:
        with pytest.raises(RuntimeError, match="GPU"):
            call()
    assert not reached
