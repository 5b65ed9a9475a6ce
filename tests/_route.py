"""Which native entry a call takes, seen on the CPU: host tensors that say they are on the device, and a library that records calls
instead of launching (or, for entries named in `real`, the library itself, whose checks run before any launch)."""
import torch

from light_vllm_amd import _mixlib, mix_ops

_load = _mixlib.load          # before a test puts a recorder in its place


class Device(torch.Tensor):
    is_cuda = property(lambda self: True)


def device(x):
    return x.as_subclass(Device)


class Recorder:
    def __init__(self, real=()):
        self.calls, self._real, self._lib = [], real, _load()

    def __getattr__(self, name):
        if name in self._real or name.endswith(("_bytes", "_error")):
            return getattr(self._lib, name)

        def call(*args):
            self.calls.append(name)
            return 0
        return call


def record(monkeypatch, real=()):
    lib = Recorder(real)
    monkeypatch.setattr(mix_ops._mixlib, "load", lambda: lib)
    monkeypatch.setattr(mix_ops, "_stream", lambda t: 0)
    return lib.calls
